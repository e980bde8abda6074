// What every Q4_0 matrix-vector kernel does with a slot (two blocks, 36 bytes): fetch it, prepare the activations it
// meets (digit planes in LDS), multiply it.  Included by the products proper (gemv_q4_0.hip) and by the launch that
// carries a whole decode step (decode_step.hip).
#pragma once
#include "common.h"
#include "gemv_xprep.h"

namespace {

struct __attribute__((aligned(4))) q4_slot {
    uint32_t w[9];  // [d0 | qs0[0..1]] [qs0 2..5] [6..9] [10..13] [qs0 14..15 | d1] [qs1 0..3] .. [qs1 12..15]
};

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// Sum over the 64 lanes of a wave; every lane ends with the total.
__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_mov<0xB1>(v);   // quad_perm(1,0,3,2)
    v += dpp_mov<0x4E>(v);   // quad_perm(2,3,0,1)
    v += dpp_mov<0x141>(v);  // row_half_mirror
    v += dpp_mov<0x140>(v);  // row_mirror
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    return v;
}

__device__ __forceinline__ float f16_bits_to_f32(uint32_t bits) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}

__device__ __forceinline__ void load_slot(q4_slot &q, const uint8_t *p) {
    const uint32_t *s = reinterpret_cast<const uint32_t *>(p);
#pragma unroll
    for (int i = 0; i < 9; i++) q.w[i] = s[i];  // plain loads: the three loads of a lane share cache lines
}

// LDS image of one prepared slot: L planes x 8 dwords, then the two block scales and the two scales of the
// blocks' corrections (0 = the block has none).  The correction planes (gemv_xprep.h) of all slots follow the
// slots: corr_dwords per slot.
template <int L>
struct slot_lds {
    static constexpr int dwords = 8 * L + 4;  // stride = 4 (mod 8): 16-byte reads of 8 lanes hit 32 distinct banks
    static constexpr int corr_dwords = 8 * xprep::CORR_L;
    static constexpr int bytes_per_slot = (dwords + corr_dwords) * 4;  // what a launch reserves per slot
};

// Sum over the 64 lanes of a wave with DPP only; the total lands in lane 63.
__device__ __forceinline__ float wave_sum_to_lane63(float v) {
    v += dpp_mov<0x111>(v);  // row_shr:1
    v += dpp_mov<0x112>(v);  // row_shr:2
    v += dpp_mov<0x114>(v);  // row_shr:4
    v += dpp_mov<0x118>(v);  // row_shr:8  -> lane 15 of each row holds the row total
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xA, 0xF, false));  // row_bcast:15
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x143, 0xC, 0xF, false));  // row_bcast:31
    return v;
}

template <int CTRL>
__device__ __forceinline__ uint32_t quad_max(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true));
}

// Eight activations of one (slot, weight-dword group) task, in the nibble order of their weight dword, to LDS:
// the L planes, the block's scale, and -- when the fixed point leaves too much of the block behind -- the
// correction planes of the residuals with their scale.  The four threads of a quad hold one block.
// refetch(y8) produces the eight activations once more: the rare path takes them from where they came from
// rather than keep them in registers past the planes, which would cost the common path its occupancy.
template <int L, class Refetch>
__device__ __forceinline__ void prep_store(const float (&x8)[8], uint32_t *slot_dst, uint32_t *corr_dst, int g,
                                           Refetch refetch) {
    // max of |x| on the bit patterns: for non-negative floats the unsigned order is the numeric
    // order, with inf and NaN on top, so a non-finite activation is never lost
    uint32_t amax = 0;
    float sum_x = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        amax = max(amax, __builtin_bit_cast(uint32_t, x8[j]) & 0x7FFFFFFFu);
        sum_x += __builtin_fabsf(x8[j]);
    }
    amax = quad_max<0xB1>(amax), sum_x += dpp_mov<0xB1>(sum_x);  // quad_perm(1,0,3,2)
    amax = quad_max<0x4E>(amax), sum_x += dpp_mov<0x4E>(sum_x);  // quad_perm(2,3,0,1)
    float mult, scale;
    xprep::block_scales<L>(amax, &mult, &scale);
    uint32_t planes[L];
    xprep::make_planes<L>(x8, mult, planes);
#pragma unroll
    for (int l = 0; l < L; l++) slot_dst[l * 8 + g] = planes[l];
    float scale2 = 0.0f;
    if (xprep::needs_correction(sum_x, amax, scale)) {  // the same in the four threads of the block; rare
        const bool no_grid = scale == 0.0f;  // every activation counts as below the top binade
        float r8[8];
        refetch(r8);
        uint32_t rmax = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t xb = __builtin_bit_cast(uint32_t, r8[j]) & 0x7FFFFFFFu;
            r8[j] = (no_grid || xprep::below_top_binade(xb, amax)) ? xprep::residual(r8[j], mult, scale) : 0.0f;
            rmax = max(rmax, __builtin_bit_cast(uint32_t, r8[j]) & 0x7FFFFFFFu);
        }
        rmax = quad_max<0xB1>(rmax);
        rmax = quad_max<0x4E>(rmax);
        float mult2;
        xprep::block_scales<xprep::CORR_L>(rmax, &mult2, &scale2);
        uint32_t planes2[xprep::CORR_L];
        xprep::make_planes<xprep::CORR_L>(r8, mult2, planes2);
#pragma unroll
        for (int l = 0; l < xprep::CORR_L; l++) corr_dst[l * 8 + g] = planes2[l];
    }
    if ((g & 3) == 0) {
        slot_dst[8 * L + (g >> 2)] = __builtin_bit_cast(uint32_t, scale);
        slot_dst[8 * L + 2 + (g >> 2)] = __builtin_bit_cast(uint32_t, scale2);
    }
}

// The eight activations of task (slot, g) of a vector in global memory, in the order prep_store takes them.
__device__ __forceinline__ void fetch_task(const float *xs /* the slot's 64 activations */, int g, float2 (&v)[4]) {
#pragma unroll
    for (int t = 0; t < 4; t += 2) {
        // nibble pairs t, t+1 of group g: weights (b, b+1) low nibbles and (16+b, 17+b) high nibbles
        const int b = xprep::group_x_index(g, 2 * t);  // even by construction
        v[t] = *reinterpret_cast<const float2 *>(xs + b);
        v[t + 1] = *reinterpret_cast<const float2 *>(xs + b + 16);
    }
}

// nibble order of the weight dword: byte b low, byte b high, byte b+1 low, byte b+1 high, ...
#define GH_TASK_X8(v) {(v)[0].x, (v)[1].x, (v)[0].y, (v)[1].y, (v)[2].x, (v)[3].x, (v)[2].y, (v)[3].y}

__device__ __forceinline__ int sdot8_first(uint32_t a, uint32_t b) {
    int d;
    asm("v_dot8_i32_i4 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b));
    return d;
}

// Integer dot of one block's four nibble dwords with the block's four dwords of each of its L planes:
// sum_l 16^l * dot8.  One accumulator per plane, issued round-robin: back-to-back v_dot8 into the same
// register serialise on the dot pipeline's latency, independent ones issue every cycle.
template <int L>
__device__ __forceinline__ int block_dot(const uint32_t (&nd)[4], const uint32_t (&xh)[L][4]) {
    int t[L];
#pragma unroll
    for (int l = 0; l < L; l++) t[l] = sdot8_first(nd[0], xh[l][0]);
#pragma unroll
    for (int i = 1; i < 4; i++)
#pragma unroll
        for (int l = 0; l < L; l++) t[l] = __builtin_amdgcn_sdot8((int)nd[i], (int)xh[l][i], t[l], false);
    int r = t[L - 1];
#pragma unroll
    for (int l = L - 2; l >= 0; l--) r = (r << 4) + t[l];
    return r;
}

// One slot of R rows: acc[r] += the dot product of row r's 64 weights (q[r]) with the slot's activations, read from
// the slot's LDS image (slot_lds) one block at a time, so that only half a slot's planes are held at once; a block
// with a correction (few, if any) also takes the same weights against its correction planes.
template <int L, int R>
__device__ __forceinline__ void slot_rows(const q4_slot (&q)[R], const uint32_t *slot_src, const uint32_t *corr_src,
                                          float *acc /* [R] */) {
    constexpr int CL = xprep::CORR_L;
    const uint32_t sign = 0x88888888u;
    const uint4 sc = *reinterpret_cast<const uint4 *>(slot_src + 8 * L);  // scales of A, B; of their corrections (0 = none)
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
        uint32_t xh[L][4];
#pragma unroll
        for (int l = 0; l < L; l++) {
            const uint4 v = *reinterpret_cast<const uint4 *>(slot_src + l * 8 + 4 * blk);
            xh[l][0] = v.x, xh[l][1] = v.y, xh[l][2] = v.z, xh[l][3] = v.w;
        }
        const float s = __builtin_bit_cast(float, blk ? sc.y : sc.x);
        const uint32_t cbits = blk ? sc.w : sc.z;
        uint32_t nd[R][4];
        float d[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (blk == 0) {
                // block A's qs start 2 bytes into the slot: each of its dwords is the top half of one word and the
                // low half of the next
                d[r] = f16_bits_to_f32(q[r].w[0] & 0xFFFFu);
#pragma unroll
                for (int i = 0; i < 4; i++) nd[r][i] = __builtin_amdgcn_alignbit(q[r].w[i + 1], q[r].w[i], 16) ^ sign;
            } else {
                d[r] = f16_bits_to_f32(q[r].w[4] >> 16);
#pragma unroll
                for (int i = 0; i < 4; i++) nd[r][i] = q[r].w[5 + i] ^ sign;
            }
            acc[r] = __builtin_fmaf(d[r] * s, (float)block_dot<L>(nd[r], xh), acc[r]);
        }
        if (cbits != 0) {
            uint32_t xc[CL][4];
#pragma unroll
            for (int l = 0; l < CL; l++) {
                const uint4 v = *reinterpret_cast<const uint4 *>(corr_src + l * 8 + 4 * blk);
                xc[l][0] = v.x, xc[l][1] = v.y, xc[l][2] = v.z, xc[l][3] = v.w;
            }
            const float s2 = __builtin_bit_cast(float, cbits);
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = __builtin_fmaf(d[r] * s2, (float)block_dot<CL>(nd[r], xc), acc[r]);
        }
    }
}

}  // namespace
