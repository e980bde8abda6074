// Q4_0 matrices against a panel of few activation rows (part of gemm_q4_0.hip).
//
// What bounds it.  Up to about a hundred rows the weights' bytes do (512 flops a byte of HBM before the matrix pipe is
// the limit), so the 256-row tile of the main kernel multiplies padding and its producer waves dequantise at the pace of
// a tile that is never full.  Here every wave dequantises its own operand in registers and no barrier stands between
// the weight stream and the matrix instructions:
//   - A wave owns NT tiles of 16 weight rows and MT tiles of 16 activation rows; a workgroup's KS waves own the same tiles
//     and take every KS-th piece of 256 k each; their sums meet in LDS at the end, in a fixed order.
//   - v_mfma_f32_16x16x32_f16 adds over k in any order as long as both operands agree on it.  Lane (r, kg) of the
//     weight operand therefore takes the whole 36-byte slot kg of the piece (two blocks of row r, as the
//     decode kernel's lanes do): one piece = eight instructions, instruction (b, c) of which multiplies the eight weights k
//     = 8c .. 8c+7 of block b of each lane's slot.  No shuffle, the block's scale is in the lane.
//   - The activation operand is then the 16-byte run c of row r in panel tile 2 kg + b: four contiguous 256-byte pieces a
//     request, from L2 (every workgroup reads the whole panel: NT rows of tiles share a fragment).
//   - The result tile has the weight rows down its registers: a lane holds four consecutive columns of Y.
// Measured (MI355X, us, weights from HBM, against the 256-row tile): see SK_MAX_ROWS.  77 rows of a 3200 x 8640 matrix through
// the f32 entry point 93 -> 17.6 to 17.9 (the generic kernel before), a prefill of 23 tokens through 32 layers 4705 -> 2490.
// Weights are rounded exactly as in the main kernel ((q - 8) * d, once, to fp16), sums are f32.
#pragma once

namespace {

constexpr int SK_PIECE = 144;  // bytes of a piece of 256 k of one row
constexpr int SK_MAX_MT = 5;  // row tiles per wave: more would take the registers of the second wave per SIMD

// How a wave's weights arrive.  SK_BLOCKS: any 2-byte aligned block, by the lane that multiplies it.  SK_SLOTS (K % 64 == 0, W
// 4-byte aligned): a 36-byte slot, likewise.  SK_RUNS (K % 256 == 0 besides): the 144 bytes a piece has of a row by a quad of
// lanes, 16 bytes each, 16 more 64 bytes on, the last 16 by the first; slots then change lanes through LDS.  A request for
// slots touches 32 to 40 lines and every line comes up in nine requests; runs are asked for once (23 rows of gate | up 20.3 ->
// 17.9 us, q | k | v of 4096 14.2 -> 11.8, each at its best tiles; which pays: skinny_pick.  Rows that are not whole pieces lose: 77 x
// 3200 x 8640 19.8 -> 21.8 with the last piece's requests moved back to the row's end).  The bits are the same.
enum sk_form { SK_BLOCKS, SK_SLOTS, SK_RUNS };
template <sk_form FORM>
struct sk_raw;

template <>
struct sk_raw<SK_SLOTS> {
    uint32_t w[9];
};
template <>
struct sk_raw<SK_RUNS> {
    uint32_t w[12];
};
template <>
struct sk_raw<SK_BLOCKS> {  // four aligned dwords and the two bytes before or behind them
    uint32_t w[2][4];
    uint32_t h[2];
};

// A piece of a tile in runs.  row: the lane's row, lane / 4 of the tile, at the lane's 16 bytes.
__device__ __forceinline__ void sk_load(sk_raw<SK_RUNS> &q, const uint8_t *row, int piece) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(row + (size_t)piece * SK_PIECE);
#pragma unroll
    for (int i = 0; i < 4; i++) q.w[i] = p[i], q.w[4 + i] = p[16 + i];
    if ((threadIdx.x & 3) == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) q.w[8 + i] = p[32 + i];
    }
}
// block: index of the lane's first block in its row (even); nblocks: blocks of the row.  Blocks past the end are
// loaded from the row's last ones and given a zero scale by sk_unpack.
__device__ __forceinline__ void sk_load(sk_raw<SK_SLOTS> &q, const uint8_t *row, int block, int nblocks) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(row + (size_t)min(block, nblocks - 2) * 18);
#pragma unroll
    for (int i = 0; i < 9; i++) q.w[i] = p[i];
}
__device__ __forceinline__ void sk_load(sk_raw<SK_BLOCKS> &q, const uint8_t *row, int block, int nblocks) {
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const uint8_t *p = row + (size_t)min(block + b, nblocks - 1) * 18;
        const bool odd = ((uintptr_t)p & 2) != 0;  // the block's d lies in front of an aligned dword: its qs are aligned
        const uint32_t *w = reinterpret_cast<const uint32_t *>(odd ? p + 2 : p);
#pragma unroll
        for (int i = 0; i < 4; i++) q.w[b][i] = w[i];
        q.h[b] = *reinterpret_cast<const uint16_t *>(odd ? p : p + 16);
    }
}

struct sk_blocks {
    uint32_t q[2][4];  // the nibble dwords of both blocks
    half2_t d[2];
};
__device__ __forceinline__ void sk_unpack_slot(sk_blocks &o, const uint32_t (&w)[9], bool in) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        o.q[0][i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], 16);
        o.q[1][i] = w[5 + i];
    }
    const _Float16 a = __builtin_bit_cast(_Float16, (uint16_t)(in ? w[0] & 0xFFFFu : 0u));
    const _Float16 b = __builtin_bit_cast(_Float16, (uint16_t)(in ? w[4] >> 16 : 0u));
    o.d[0] = half2_t{a, a}, o.d[1] = half2_t{b, b};
}
__device__ __forceinline__ void sk_unpack(sk_blocks &o, const sk_raw<SK_SLOTS> &r, int block, int nblocks) {
    sk_unpack_slot(o, r.w, block < nblocks);
}
// lds: the wave's own 2304 bytes, the tile's rows one behind the other.
__device__ __forceinline__ void sk_unpack(sk_blocks &o, const sk_raw<SK_RUNS> &r, uint8_t *lds) {
    const int lane = threadIdx.x & 63;
    uint8_t *put = lds + (lane >> 2) * SK_PIECE + (lane & 3) * 16;
    *reinterpret_cast<uint4 *>(put) = make_uint4(r.w[0], r.w[1], r.w[2], r.w[3]);
    *reinterpret_cast<uint4 *>(put + 64) = make_uint4(r.w[4], r.w[5], r.w[6], r.w[7]);
    if ((lane & 3) == 0) *reinterpret_cast<uint4 *>(put + 128) = make_uint4(r.w[8], r.w[9], r.w[10], r.w[11]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // (a wave's LDS instructions execute in order)
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint32_t *get = reinterpret_cast<const uint32_t *>(lds) + (lane & 15) * (SK_PIECE / 4) + (lane >> 4) * 9;
    uint32_t w[9];
#pragma unroll
    for (int i = 0; i < 9; i++) w[i] = get[i];  // 36 bytes from lane to lane: no two lanes in one bank
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    sk_unpack_slot(o, w, true);
}
__device__ __forceinline__ void sk_unpack(sk_blocks &o, const sk_raw<SK_BLOCKS> &r, const uint8_t *row, int block, int nblocks) {
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const bool odd = ((uintptr_t)(row + (size_t)min(block + b, nblocks - 1) * 18) & 2) != 0;
        const uint32_t next[4] = {r.w[b][1], r.w[b][2], r.w[b][3], r.h[b]};
#pragma unroll
        for (int i = 0; i < 4; i++) o.q[b][i] = odd ? r.w[b][i] : __builtin_amdgcn_alignbit(next[i], r.w[b][i], 16);
        const uint32_t bits = odd ? r.h[b] : r.w[b][0] & 0xFFFFu;
        const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)(block + b < nblocks ? bits : 0u));
        o.d[b] = half2_t{d, d};
    }
}

// Weights k = 8c .. 8c+7 of a block as fp16: the low (c < 2) or high nibbles of the dwords 2 (c % 2) and 2 (c % 2) + 1.
template <int C>
__device__ __forceinline__ half8_t sk_operand(const uint32_t (&q)[4], half2_t d) {
    const half2_t off = {(_Float16)1032.0f, (_Float16)1032.0f};
    uint4 o;
    uint32_t *ov = &o.x;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t v = q[2 * (C & 1) + i];
        const uint32_t n = (C < 2 ? v : v >> 4) & 0x0F0F0F0Fu;
        // 0x64nn is 1024 + nn: minus 1032 the exact integer n - 8, rounded once by the product with d
        const half2_t a = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, n, 0x04010400u));
        const half2_t b = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, n, 0x04030402u));
        ov[2 * i] = __builtin_bit_cast(uint32_t, (a - off) * d);
        ov[2 * i + 1] = __builtin_bit_cast(uint32_t, (b - off) * d);
    }
    return __builtin_bit_cast(half8_t, o);
}

// Instructions of a piece whose activation fragments are requested together: about eight fragments in flight a wave.  Two and four
// weight tiles under four row tiles have half as many where weights come in runs: 4 x 4 spilled five registers with two instructions'
// (56 x 4096 x 14000 22.5 -> 22.0 us, 64 x 1024 x 16384 11.9 -> 11.1); 2 x 4, chosen from K = 8192 on, took 173, a wave per SIMD less
// than in slots, and takes 141 (64 x 11008 x 6848 31.8 -> 29.8 us, 52 x 8192 x 6752 24.5 -> 23.2; 28 sizes 4.7 to 6.3 % less).
constexpr int sk_steps(int nt, int mt, sk_form form) {
    return mt <= 1 ? 4 : mt <= (nt % 2 == 0 && form == SK_RUNS ? 3 : 4) ? 2 : 1;
}
// Waves per SIMD the registers are kept to: four hide the requests' latency where the tiles allow it (2 x 2 tiles: 138 -> 110
// registers, gate | up at 23 rows 21.4 -> 20.3 us with weights in the Infinity Cache, 25.2 from HBM).
constexpr int sk_occ(int nt, int mt, sk_form form) {
    const int regs = 4 * nt * mt + 8 * sk_steps(nt, mt, form) * mt + (form == SK_RUNS ? 22 : 19) * nt + 40;
    return regs <= 138 ? 4 : regs <= 175 ? 3 : 2;
}

// Where four consecutive columns of row m go: n is a column of the concatenated matrices.
template <typename MATS>
__device__ __forceinline__ void sk_store4(const MATS &mats, int n, int m, float4_t v) {
    if (n >= mats.n_total) return;
    float *Y = mats.Y[0];
    int N = mats.N[0], first = 0;
#pragma unroll
    for (int t = 1; t < GEMM_MAX_MATS; t++) {
        const bool ge = n >= mats.col0[t];
        Y = ge ? mats.Y[t] : Y, N = ge ? mats.N[t] : N, first = ge ? mats.col0[t] : first;
    }
    if constexpr (gemm_has_rope<MATS>) {  // q | k | v: every matrix has whole sixteens of columns, its rows are 16-byte aligned
        if (n < mats.col0[2]) {
            const float4 cs = *reinterpret_cast<const float4 *>(mats.rope + (size_t)m * 64 + (((n - first) & 127) >> 1));
            const float2 c0 = make_float2(cs.x, cs.y), c1 = make_float2(cs.z, cs.w);
            v = float4_t{gemm_rotate(v[0], v[1], c0, false), gemm_rotate(v[1], v[0], c0, true), gemm_rotate(v[2], v[3], c1, false),
                         gemm_rotate(v[3], v[2], c1, true)};
        }
        if (mats.kv_f16 && n >= mats.col0[1]) {
            asm volatile("" : "+v"(v));  // rounded to f32 first, as the ops one by one would
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            *reinterpret_cast<h4 *>(reinterpret_cast<_Float16 *>(Y) + (size_t)m * N + (n - first)) =
                h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
            return;
        }
    }
    float *dst = Y + (size_t)m * N + (n - first);
    if (n - first + 4 <= N && ((uintptr_t)dst & 15) == 0) {
        *reinterpret_cast<float4_t *>(dst) = v;
        return;
    }
    for (int e = 0; e < 4; e++) {  // a ragged or unaligned result, or four columns that go on in the next matrix
        const int ne = n + e;
        if (ne >= mats.n_total) return;
        Y = mats.Y[0], N = mats.N[0], first = 0;
        for (int t = 1; t < GEMM_MAX_MATS; t++)
            if (ne >= mats.col0[t]) Y = mats.Y[t], N = mats.N[t], first = mats.col0[t];
        Y[(size_t)m * N + (ne - first)] = v[e];
    }
}

// K: the rows' true length (a multiple of 32); kp_blocks: 32-k blocks of a panel row, a multiple of 8, zeros past K.
// With mats.swiglu_out the first NT / 2 tiles are gate rows and the others the same rows of the up matrix.
template <int NT, int MT, int KS, sk_form FORM, typename MATS>
__global__ __launch_bounds__(KS * 64, sk_occ(NT, MT, FORM)) void gemm_q4_0_skinny(const MATS mats, const _Float16 *__restrict__ Xh, int K,
                                                            int kp_blocks, int M, int n_tiles, int m_blocks) {
    constexpr int SG = sk_steps(NT, MT, FORM), GROUPS = 8 / SG;  // an even number of groups a piece
    __shared__ __attribute__((aligned(16))) float4_t part[KS][KS][64];
    static_assert(sizeof(part[0]) >= 16 * SK_PIECE, "a wave's tile of weights lies in its share of the sums' LDS");
    // blockIdx % 8 is the XCD: the row blocks of one weight tile follow one another on it, so the second reads its
    // weights from that XCD's L2
    const int idx = blockIdx.x >> 3;
    const int nt0 = (idx / m_blocks) * 8 + (blockIdx.x & 7), mb = idx % m_blocks;
    if (nt0 >= n_tiles) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, kg = lane >> 4, wr = FORM == SK_RUNS ? lane >> 2 : r;  // wr: the row whose weights the lane requests
    uint8_t *const wlds = reinterpret_cast<uint8_t *>(part[wave]);
    const bool swiglu = mats.swiglu_out != nullptr;
    const int nblocks = K / 32, npieces = kp_blocks / 8;
    const size_t wrow_bytes = (size_t)nblocks * 18;

    const uint8_t *row[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        if (NT > 1 && swiglu)
            row[t] = mats.W[t >= NT / 2] + (size_t)min(nt0 * (NT / 2 * 16) + (t % (NT / 2 > 0 ? NT / 2 : 1)) * 16 + wr, mats.N[0] - 1) * wrow_bytes;
        else
            row[t] = gemm_w_row(mats, nt0 * (NT * 16) + t * 16 + wr, wrow_bytes);
    }
    // fragment (b, c) of row tile i, piece p: byte fo[i] + p * 8 KB + b * 1 KB + c * 256 of the panel
    const int m16_last = (M + 15) / 16 - 1;
    uint32_t fo[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) fo[i] = (uint32_t)min(mb * MT + i, m16_last) * (uint32_t)kp_blocks * 1024u + kg * 2048u + r * 16u;

    float4_t acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[t][i] = float4_t{0.f, 0.f, 0.f, 0.f};

    const unsigned char *xb = reinterpret_cast<const unsigned char *>(Xh);
    half8_t f[2][SG][MT];
    auto frags = [&](half8_t(&dst)[SG][MT], int piece, int g) {
#pragma unroll
        for (int j = 0; j < SG; j++)
#pragma unroll
            for (int i = 0; i < MT; i++)
                dst[j][i] = *reinterpret_cast<const half8_t *>(xb + (size_t)piece * 8192 + fo[i] + (g * SG + j) / 4 * 1024 + (g * SG + j) % 4 * 256);
    };
    sk_raw<FORM> raw[NT];
    auto weights = [&](sk_raw<FORM> &q, const uint8_t *w, int p) {
        if constexpr (FORM == SK_RUNS)
            sk_load(q, w + (lane & 3) * 16, p);
        else
            sk_load(q, w, p * 8 + kg * 2, nblocks);
    };
    int piece = wave;
    if (piece < npieces) {
#pragma unroll
        for (int t = 0; t < NT; t++) weights(raw[t], row[t], piece);
        frags(f[0], piece, 0);
    }
    for (; piece < npieces; piece += KS) {
        const int next = min(piece + KS, npieces - 1);  // the last round requests a piece again, unused
        sk_blocks blk[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if constexpr (FORM == SK_RUNS)
                sk_unpack(blk[t], raw[t], wlds);
            else if constexpr (FORM == SK_SLOTS)
                sk_unpack(blk[t], raw[t], piece * 8 + kg * 2, nblocks);
            else
                sk_unpack(blk[t], raw[t], row[t], piece * 8 + kg * 2, nblocks);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NT; t++) weights(raw[t], row[t], next);
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
            frags(f[(g + 1) & 1], g + 1 < GROUPS ? piece : next, (g + 1) % GROUPS);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < SG; j++) {
                const int step = g * SG + j, b = step / 4;
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    const half8_t w = step % 4 == 0   ? sk_operand<0>(blk[t].q[b], blk[t].d[b])
                                      : step % 4 == 1 ? sk_operand<1>(blk[t].q[b], blk[t].d[b])
                                      : step % 4 == 2 ? sk_operand<2>(blk[t].q[b], blk[t].d[b])
                                                      : sk_operand<3>(blk[t].q[b], blk[t].d[b]);
#pragma unroll
                    for (int i = 0; i < MT; i++) acc[t][i] = GEMM_MFMA(w, f[g & 1][j][i], acc[t][i]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // The waves' sums, KS tiles at a time: every wave parks its own, then adds up one of them.  Tiles go in the order
    // (i, t), for a SwiGLU with the gate and the up tile of an output next to each other.
    constexpr int TILES = NT * MT;
#pragma unroll
    for (int c0 = 0; c0 < TILES; c0 += KS) {
        if (c0 || FORM == SK_RUNS) __syncthreads();  // (the waves' weights lie where the first sums go)
#pragma unroll
        for (int j = 0; j < KS; j++) {
            constexpr int H = NT / 2 > 0 ? NT / 2 : 1;
            if (c0 + j < TILES) {
                const int i = (c0 + j) / NT, o = (c0 + j) % NT;
                const int t_pair = (o & 1) * H + (o >> 1);  // gate 0, up 0, gate 1, up 1 ..
                part[j][wave][lane] = NT > 1 && swiglu ? acc[t_pair][i] : acc[o][i];
            }
        }
        __syncthreads();
        const int j = wave;
        const int tile = c0 + j;
        const int i = tile / NT, o = tile % NT;
        const int m = (mb * MT + i) * 16 + r;
        if (tile >= TILES) continue;
        float4_t v = part[j][0][lane];
#pragma unroll
        for (int w = 1; w < KS; w++) v += part[j][w][lane];
        if (NT > 1 && swiglu) {
            if (o & 1) continue;  // the up tile is read by the wave of its gate tile
            float4_t u = part[j + 1 < KS ? j + 1 : j][0][lane];
#pragma unroll
            for (int w = 1; w < KS; w++) u += part[j + 1 < KS ? j + 1 : j][w][lane];
            const int n = nt0 * (NT / 2 * 16) + (o >> 1) * 16 + 4 * kg;
            const int N = mats.N[0];
            if (m < ((M + 15) & ~15) && n < N) {  // rows past M are zeros in the input panel, hence here
                float s[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float sig = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(v[e] * -1.44269504088896340736f));
                    s[e] = (v[e] * sig) * u[e];
                }
                unsigned char *out = reinterpret_cast<unsigned char *>(mats.swiglu_out) + (size_t)(m >> 4) * (size_t)(N >> 5) * 1024 +
                                     (size_t)(n >> 5) * 1024 + (size_t)((n & 31) >> 3) * 256 + (size_t)(m & 15) * 16 + (size_t)(n & 7) * 2;
                *reinterpret_cast<uint2 *>(out) = make_uint2(pack_h2(s[0], s[1]), pack_h2(s[2], s[3]));
            }
        } else if (m < M) {
            sk_store4(mats, nt0 * (NT * 16) + o * 16 + 4 * kg, m, v);
        }
    }
}

template <int NT, int MT, int KS, sk_form FORM, typename MATS>
int32_t skinny_launch(galois_hip_ctx *ctx, const MATS &mats, const _Float16 *Xh, int K, int kp_blocks, int M) {
    const int cols_per_tile = mats.swiglu_out ? NT / 2 * 16 : NT * 16;
    const int cols = mats.swiglu_out ? mats.N[0] : mats.n_total;
    const int n_tiles = (cols + cols_per_tile - 1) / cols_per_tile, m_blocks = ((M + 15) / 16 + MT - 1) / MT;
    const dim3 grid((unsigned)((n_tiles + 7) / 8 * 8 * m_blocks));
    hipLaunchKernelGGL((gemm_q4_0_skinny<NT, MT, KS, FORM, MATS>), grid, dim3(KS * 64), 0, ctx->stream, mats, Xh, K, kp_blocks, M,
                       n_tiles, m_blocks);
    return GALOIS_HIP_OK;
}

// Rows up to which the panel calls run here rather than on the wide kernel.  Measured (us, this kernel / that one at its best
// tile, weights from HBM): q | k | v of 4096 (12288 x 4096) 16.5 / 20.6 at 23 rows, 19.9 / 21.2 at 64, 22.4 / 21.7 at 80, 29.9 / 21.8 at
// 100; gate | up + SwiGLU (2 x 11008 x 4096) 25.2 / 31.8, 33.5 / 33.2, 35.9 / 33.2, 43.5 / 32.8; of models 1024 wide 5.5 / 7.8 and 6.0 /
// 11.6 at 80 rows, 5.6 / 7.9 and 8.0 / 11.6 at 100.  Narrow matrices stay ahead here for longer (11008 -> 4096 at 150 rows 27 / 39 in
// shares), which gemm_pick_form uses where a caller lets the sums take any order.  In the panel calls without that freedom, and in
// the f32 entry point up to this line, the order of a result's sum depends on K and on the side of this line M is on, never on N, so
// matrices multiplied together, one by one or with the SwiGLU behind them give the same bits (above it the f32 entry point may take
// two shares of k by N).
constexpr int SK_MAX_ROWS = 80;

// Time of a workgroup relative to others, us at K = 4096 (fitted within 10 %): what a weight tile costs
// (its bytes, its dequantisation), what a row tile costs (its fragments) and their products.  runs: by the form of the weights.
// One weight tile under many row tiles gains nothing from runs at eight waves (40 x 11008 x 4096: 1 x 3 tiles 22.3 us in slots, 23.1 in
// runs, 2 x 2 20.4).
inline double sk_cost(int nt, int mt, bool runs, int K) {
    if (runs) return nt == 1 ? 2.0 + (K >= 8192 && mt >= 3 ? 1.25 : 1.12) * mt : nt == 2 ? 3.6 + 1.05 * mt : nt == 3 ? 5.0 + 1.3 * mt : 6.5 + 1.72 * mt;
    return 1.55 * nt + mt * (0.78 + 0.25 * nt);
}

template <int KS, sk_form FORM, typename MATS>
int32_t skinny_launch_tiles(galois_hip_ctx *ctx, const MATS &mats, const _Float16 *Xh, int K, int kp_blocks, int M, int nt, int mt) {
#define SK_MT(NT_)                                                                                    \
    switch (mt) {                                                                                     \
        case 1: return skinny_launch<NT_, 1, KS, FORM>(ctx, mats, Xh, K, kp_blocks, M);            \
        case 2: return skinny_launch<NT_, 2, KS, FORM>(ctx, mats, Xh, K, kp_blocks, M);            \
        case 3: return skinny_launch<NT_, 3, KS, FORM>(ctx, mats, Xh, K, kp_blocks, M);            \
        case 4: return skinny_launch<NT_, 4, KS, FORM>(ctx, mats, Xh, K, kp_blocks, M);            \
        default: return skinny_launch<NT_, SK_MAX_MT, KS, FORM>(ctx, mats, Xh, K, kp_blocks, M);   \
    }
    if (nt == 1) SK_MT(1)
    if (nt == 2) SK_MT(2)
    if (nt == 3) SK_MT(3)
    SK_MT(4)
#undef SK_MT
}

// Tiles per wave by that cost and the rounds of workgroups over the CUs; the rows may be split over several workgroups.
struct sk_tiles {
    int nt, mt;
    double cost;
    bool runs;
};
// whole: the weights' rows are whole pieces and 4-byte aligned, so that runs are possible.
inline sk_tiles skinny_pick(const galois_hip_ctx *ctx, int64_t cols, int K, int M, bool swiglu, bool whole) {
    const int64_t cus = ctx->n_cu > 0 ? ctx->n_cu : 256;
    const int t = (M + 15) / 16;
    sk_tiles best = {0, 0, 0.0, false};
    for (int m = 1; m <= SK_MAX_MT && m <= t; m++)
        for (int n = swiglu ? 2 : 1; n <= 4; n += swiglu ? 2 : 1) {
            // three tiles a wave fill the device where two leave a second round nearly empty (77 x 3200 x 8640: 180 workgroups
            // instead of 270 or 135; 12288 columns: 256); not where that splits rows that one workgroup could take, unless they are long and come in
            // runs (72 x 1408 x 4183 11.8 us as two blocks of 3 x 3 tiles, 11.0 as one of 2 x 5; 74 x 4000 x 5277 17.3 / 16.4; 80 x 768 x 5463 9.7 /
            // 9.1; but 80 x 2048 x 5632 11.4 / 12.0, 56 x 11008 x 5120 27.0 / 30.9).  Short rows are better off in more rounds (beyond 80 rows up to K = 1216: 177 x 1216 x 6951 16.6 us in
            // three tiles, 15.9 without; 355 x 608 x 4533 16.0, 14.5), up to sixteen rows the longer the fewer columns there are (us in three tiles / in one: 16 x 3328 x 9216 12.6 / 11.4,
            // x 12288 13.8 / 13.7; 16 x 3584 x 10240 12.7 / 11.9, x 12288 14.3 / 15.3; 16 x 4096 x 8640 12.7 / 12.1, x 11008 14.3 / 15.7; 16 x 4352 x
            // 8640 14.0 / 13.1, x 9216 14.8 / 14.9)
            if (n == 3 && ((m < t && t <= SK_MAX_MT && (!whole || K < 2048)) ||
                           (m > 1 ? K <= (t <= SK_MAX_MT ? 512 : 1216) : K <= 2560 || (double)cols < (double)cus * (37.0 + (4352 - K) * 3 / 256.0))))
                continue;
            const int64_t tiles = (cols + 16 * n - 1) / (16 * n), blocks = (t + m - 1) / m;
            // The weight tiles are dealt to eight XCDs (blockIdx % 8), so a launch runs as long as its fullest XCD, which may hold
            // more workgroups than CUs where the device as a whole does not (524 x 8192 x 1792: 28 tiles of nine row blocks,
            // 36 workgroups on four of the XCDs, 52 us against 32 with other tiles).  With very many rows that evens out.
            const int64_t wgs = (t < 64 ? (tiles + 7) / 8 * 8 : tiles) * blocks;
            // Runs pay where a CU has more to do than one workgroup's chain of requests, whose LDS trip they lengthen: long rows
            // (eight waves), a second workgroup, three or four weight tiles a wave (over 500 sizes 3 to 6 % each; elsewhere -3 to 0 %); not with
            // two pieces a row, a wave's only one (3 x 512 x 8653 6.9 us in runs, 6.7 in slots).
            // Workgroups that share a CU then overlap a little.
            double rounds = (double)((wgs + cus - 1) / cus);
            // Four by four tiles have fewer fragments in flight with runs than with slots, which costs more than it gains where four
            // waves have long rows (64 x 4608 x 14500 24.3 us in runs, 25.2 in slots, x 7424 35.5 / 34.4; eight waves, x 9472 38.7 / 40.6).
            const bool runs = whole && K > 512 && (K >= 8192 || wgs > cus || n >= 3) && !(n == 4 && m == 4 && K > 5120 && K < 8192);
            const double cost = rounds * (runs && K < 8192 && rounds > 1 ? rounds > 2 ? 0.85 : 0.9 : 1.0) * sk_cost(n, m, runs, K);
            if (best.nt == 0 || cost < best.cost) best = {n, m, cost, runs};
        }
    return best;
}
inline double sk_far(const sk_tiles &t, int M) {  // row blocks past what shares a weight tile's panel traffic, 0 .. 1
    const double blocks = (double)(((int64_t)M + 15) / 16 / t.mt);
    return blocks <= 12.0 ? 0.0 : blocks < 28.0 ? (blocks - 12.0) / 16.0 : 1.0;
}
// Over 2652 sizes (K 512 .. 11008, N 512 .. 5120, 81 .. 2000 rows) within 10 %.
inline double skinny_us(const galois_hip_ctx *ctx, int N, int K, int M) {
    const sk_tiles t = skinny_pick(ctx, N, K, M, false, true);
    return 1.0 + 1.05 * t.cost * K / 4096.0 * (1.0 + 0.3 * sk_far(t, M));
}

// KS by K alone (the order of the sums): eight waves for long rows, whose pieces keep them busy.  t: tiles the caller has picked.
template <typename MATS>
int32_t skinny_launch_any(galois_hip_ctx *ctx, const MATS &mats, const _Float16 *Xh, int K, int kp_blocks, int M, bool aligned,
                          sk_tiles t = {0, 0, 0.0, false}) {
    const bool swiglu = mats.swiglu_out != nullptr;
    if (t.nt == 0) t = skinny_pick(ctx, swiglu ? 2 * (int64_t)mats.N[0] : mats.n_total, K, M, swiglu, aligned && K % 256 == 0);
    const sk_form form = !aligned ? SK_BLOCKS : t.runs ? SK_RUNS : SK_SLOTS;
    constexpr sk_form other = gemm_has_rope<MATS> ? SK_SLOTS : SK_BLOCKS;  // q | k | v with their rotation are aligned
    GH_REQUIRE(ctx, form != SK_BLOCKS || other == SK_BLOCKS, GALOIS_HIP_E_ALIGN, "matmul: rotation behind unaligned weights");
#define SK_FORM(KS_)                                                                                                     \
    return form == SK_RUNS    ? skinny_launch_tiles<KS_, SK_RUNS>(ctx, mats, Xh, K, kp_blocks, M, t.nt, t.mt)            \
           : form == SK_SLOTS ? skinny_launch_tiles<KS_, SK_SLOTS>(ctx, mats, Xh, K, kp_blocks, M, t.nt, t.mt)           \
                              : skinny_launch_tiles<KS_, other>(ctx, mats, Xh, K, kp_blocks, M, t.nt, t.mt)
    if (K >= 8192) SK_FORM(8);
    SK_FORM(4);
#undef SK_FORM
}

}  // namespace
