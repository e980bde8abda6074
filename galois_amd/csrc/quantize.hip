// f32 -> Q4_0 quantizer on the device.
//
// galois leaves BlockQ4_0::from_f32 as todo!() (src/ggml_quants.rs:198-200); Q4_0 data
// reaches it as ready-made bytes (src/lib.rs:2477-2491).  This kernel produces those bytes
// with the canonical ggml rule so that to_f32 (src/ggml_quants.rs:209-228) inverts them:
// per block of 32 the element of largest magnitude (first wins) fixes d = max / -8,
// id = 1/d (0 when d == 0) from the unrounded f32 d, q = min(15, trunc(x*id + 8.5)).
// Every operation is a separately rounded IEEE f32 operation (no fused multiply-add), so
// the bytes are identical to a CPU evaluation of the same rule.
#include "common.h"

namespace {

__global__ __launch_bounds__(256) void quantize_q4_0_blocks(const float *__restrict__ x, uint16_t *__restrict__ y,
                                                           int64_t nblocks) {
#pragma clang fp contract(off)  // the rule is defined with separately rounded multiply and add
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (b >= nblocks) return;
    const float *xb = x + b * 32;
    float v[32];
#pragma unroll
    for (int j = 0; j < 32; j++) v[j] = xb[j];
    float amax = 0.0f, mx = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; j++) {
        const float a = __builtin_fabsf(v[j]);
        if (amax < a) {
            amax = a;
            mx = v[j];
        }
    }
    float d = mx * -0.125f;  // == mx / -8 exactly (power of two), keeps the sign of zero
    // keep the product a value of its own: fused into the f16 conversion it would be formed as
    // mx * -0.125 + 0, and (-0) + (+0) loses the sign of an all-zero block's scale
    asm volatile("" : "+v"(d));
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    uint16_t *out = y + b * 9;
    out[0] = __builtin_bit_cast(uint16_t, (_Float16)d);
#pragma unroll
    for (int j = 0; j < 16; j += 2) {
        uint32_t bytes = 0;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int q0 = (int)(v[j + t] * id + 8.5f);
            const int q1 = (int)(v[j + t + 16] * id + 8.5f);
            bytes |= (uint32_t)(min(q0, 15) | (min(q1, 15) << 4)) << (8 * t);
        }
        out[1 + j / 2] = (uint16_t)bytes;
    }
}

// Both directions for 16-byte aligned arrays.  A pass over HBM and nothing else: a thread per block (above, below) makes
// every request of a wave touch 64 lines 128 bytes apart on the f32 side and writes the 18-byte side in 2-byte pieces;
// here eight lanes share a block, four consecutive floats each, so a wave's requests on the f32 side are one contiguous
// KB, and the blocks pass through LDS (128 of them, 2304 bytes, a workgroup) in 16-byte pieces.  Measured on 11008 x 4096
// (206 MB a direction): quantize 46.2 -> 34.4 us, dequantize 56.9 -> 29.4 us.
constexpr int QB = 128;                // blocks per workgroup
constexpr int QB_CHUNKS = QB * 18 / 16;  // 16-byte pieces of them
typedef float float4_t __attribute__((ext_vector_type(4)));

// Exchanges between the eight lanes of a block, on the vector pipe: as shuffles through LDS, and with a division per lane and
// block, they made the kernel slower than a thread per block on inputs that are in a cache (131072 blocks: thread per
// block 4.1 us, shuffles 4.9, this 4.0; 300000 blocks 8.6, 9.8, 8.3; from HBM 10.9, 11.2, 9.7).
enum { QZ_SWAP1 = 0xB1, QZ_SWAP2 = 0x4E, QZ_REVERSE = 0x1B, QZ_HALF_MIRROR = 0x141 };  // quad_perm 1032, 2301, 3210; lane 7 - g
template <int CTRL>
__device__ __forceinline__ float qz_dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ void qz_first_max(float &amax, float &mx, bool upper) {
    const float oa = qz_dpp<CTRL>(amax), om = qz_dpp<CTRL>(mx);
    const bool take = upper ? oa >= amax : oa > amax;
    amax = take ? oa : amax, mx = take ? om : mx;
}

__global__ __launch_bounds__(256) void quantize_q4_0_lanes(const float4_t *__restrict__ x, uint8_t *__restrict__ y, int64_t nblocks) {
#pragma clang fp contract(off)  // as above
    __shared__ __attribute__((aligned(16))) uint8_t out[QB * 18];
    const int64_t b0 = (int64_t)blockIdx.x * QB;
    const int nb = (int)(nblocks - b0 < QB ? nblocks - b0 : QB);
    const int g = threadIdx.x & 7, bl = threadIdx.x >> 3;  // elements 4g .. 4g+3 of blocks bl, bl + 32, ..
    float4_t v[QB / 32];
#pragma unroll
    for (int i = 0; i < QB / 32; i++) v[i] = x[(b0 + (bl + 32 * i < nb ? bl + 32 * i : nb - 1)) * 8 + g];
    float mx[QB / 32];
#pragma unroll
    for (int i = 0; i < QB / 32; i++) {
        float amax = 0.0f;
        mx[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float a = __builtin_fabsf(v[i][j]);
            if (amax < a) amax = a, mx[i] = v[i][j];
        }
        // the block's first element of largest magnitude: at equal magnitude the lower lane's
        qz_first_max<QZ_SWAP1>(amax, mx[i], g & 1);
        qz_first_max<QZ_SWAP2>(amax, mx[i], g & 2);
        qz_first_max<QZ_HALF_MIRROR>(amax, mx[i], g & 4);  // the four lanes of a quad agree by now
    }
    // lane g works out the scale of block g % 4 of the lane's four, and the quad passes it round: one division instead of four
    static_assert(QB / 32 == 4, "four blocks a lane, four lanes a quad");
    const float mxs = (g & 2) ? ((g & 1) ? mx[3] : mx[2]) : ((g & 1) ? mx[1] : mx[0]);
    float d = mxs * -0.125f;
    asm volatile("" : "+v"(d));
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    if (g >= 4) *reinterpret_cast<uint16_t *>(out + (bl + 32 * (g - 4)) * 18) = __builtin_bit_cast(uint16_t, (_Float16)d);
    const float ids[4] = {qz_dpp<0x00>(id), qz_dpp<0x55>(id), qz_dpp<0xAA>(id), qz_dpp<0xFF>(id)};
#pragma unroll
    for (int i = 0; i < QB / 32; i++) {
        uint32_t nib = 0;  // one value per byte
#pragma unroll
        for (int j = 0; j < 4; j++) nib |= (uint32_t)(min((int)(v[i][j] * ids[i] + 8.5f), 15) & 15) << (8 * j);
        // lane g + 4 holds elements 16 + 4g ..: the high nibbles of the same bytes (its quad reversed, then the eight lanes)
        const uint32_t high = __builtin_bit_cast(uint32_t, qz_dpp<QZ_HALF_MIRROR>(qz_dpp<QZ_REVERSE>(__builtin_bit_cast(float, nib))));
        uint16_t *o = reinterpret_cast<uint16_t *>(out + (bl + 32 * i) * 18);
        if (g < 4) {
            const uint32_t q = nib | high << 4;
            o[1 + 2 * g] = (uint16_t)q, o[2 + 2 * g] = (uint16_t)(q >> 16);
        }
    }
    __syncthreads();
    uint8_t *dst = y + b0 * 18;
    const int bytes = nb * 18;
    for (int c = threadIdx.x; c < QB_CHUNKS; c += 256) {
        if (c * 16 + 16 <= bytes)
            reinterpret_cast<uint4 *>(dst)[c] = reinterpret_cast<const uint4 *>(out)[c];
        else
            for (int t = c * 16; t < bytes; t += 2) *reinterpret_cast<uint16_t *>(dst + t) = *reinterpret_cast<const uint16_t *>(out + t);
    }
}

__global__ __launch_bounds__(256) void dequantize_q4_0_lanes(const uint8_t *__restrict__ x, float4_t *__restrict__ y, int64_t nblocks) {
    __shared__ __attribute__((aligned(16))) uint8_t in[QB * 18];
    const int64_t b0 = (int64_t)blockIdx.x * QB;
    const int nb = (int)(nblocks - b0 < QB ? nblocks - b0 : QB);
    const uint8_t *src = x + b0 * 18;
    const int bytes = nb * 18;
    for (int c = threadIdx.x; c < QB_CHUNKS; c += 256) {
        if (c * 16 + 16 <= bytes)
            reinterpret_cast<uint4 *>(in)[c] = reinterpret_cast<const uint4 *>(src)[c];
        else
            for (int t = c * 16; t < bytes; t += 2) *reinterpret_cast<uint16_t *>(in + t) = *reinterpret_cast<const uint16_t *>(src + t);
    }
    __syncthreads();
    const int g = threadIdx.x & 7, bl = threadIdx.x >> 3, shift = g < 4 ? 0 : 4;
#pragma unroll
    for (int i = 0; i < QB / 32; i++) {
        const int b = bl + 32 * i;
        if (b >= nb) break;
        const uint16_t *p = reinterpret_cast<const uint16_t *>(in + b * 18);
        const float d = (float)__builtin_bit_cast(_Float16, p[0]);
        const uint32_t q = (p[1 + 2 * (g & 3)] | (uint32_t)p[2 + 2 * (g & 3)] << 16) >> shift;  // bytes 4 (g % 4) ..
        float4_t o;
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = (float)((int)((q >> (8 * j)) & 0xF) - 8) * d;
        __builtin_nontemporal_store(o, y + (b0 + b) * 8 + g);
    }
}

// to_f32 (src/ggml_quants.rs:209-228): blocks -> f32, exact.
__global__ __launch_bounds__(256) void dequantize_q4_0_blocks(const uint16_t *__restrict__ x, float *__restrict__ y,
                                                             int64_t nblocks) {
    const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (b >= nblocks) return;
    const uint16_t *p = x + b * 9;
    const float d = (float)__builtin_bit_cast(_Float16, p[0]);
    float *out = y + b * 32;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const uint32_t v = p[1 + j];
        out[2 * j] = (float)((int)(v & 0xF) - 8) * d;
        out[2 * j + 16] = (float)((int)((v >> 4) & 0xF) - 8) * d;
        out[2 * j + 1] = (float)((int)((v >> 8) & 0xF) - 8) * d;
        out[2 * j + 17] = (float)((int)((v >> 12) & 0xF) - 8) * d;
    }
}

}  // namespace

extern "C" {

int32_t galois_hip_quantize_row_q4_0(galois_hip_ctx *ctx, const float *x, void *y, int64_t k) {
    GH_REQUIRE_CTX(ctx);
    GH_REQUIRE(ctx, x && y, GALOIS_HIP_E_NULL, "quantize_row_q4_0");
    GH_REQUIRE(ctx, k > 0 && k % 32 == 0 && k / 32 <= (int64_t)0x7FFFFFFF * 256, GALOIS_HIP_E_SHAPE,
               "quantize_row_q4_0: k must be a positive multiple of 32");
    GH_REQUIRE(ctx, gh_aligned(x, 4) && gh_aligned(y, 2), GALOIS_HIP_E_ALIGN, "quantize_row_q4_0");
    GH_BIND(ctx);
    const int64_t nb = k / 32;
    if (gh_aligned(x, 16) && gh_aligned(y, 16) && nb / QB < 0x7FFFFFFF)
        hipLaunchKernelGGL(quantize_q4_0_lanes, dim3((unsigned)((nb + QB - 1) / QB)), dim3(256), 0, ctx->stream,
                           reinterpret_cast<const float4_t *>(x), (uint8_t *)y, nb);
    else
        hipLaunchKernelGGL(quantize_q4_0_blocks, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, ctx->stream, x,
                           (uint16_t *)y, nb);
    GH_LAUNCH_CHECK(ctx, "quantize_row_q4_0 launch");
}

int32_t galois_hip_dequantize_row_q4_0(galois_hip_ctx *ctx, const void *x, float *y, int64_t k) {
    GH_REQUIRE_CTX(ctx);
    GH_REQUIRE(ctx, x && y, GALOIS_HIP_E_NULL, "dequantize_row_q4_0");
    GH_REQUIRE(ctx, k > 0 && k % 32 == 0 && k / 32 <= (int64_t)0x7FFFFFFF * 256, GALOIS_HIP_E_SHAPE,
               "dequantize_row_q4_0: k must be a positive multiple of 32");
    GH_REQUIRE(ctx, gh_aligned(x, 2) && gh_aligned(y, 4), GALOIS_HIP_E_ALIGN, "dequantize_row_q4_0");
    GH_BIND(ctx);
    const int64_t nb = k / 32;
    if (gh_aligned(x, 16) && gh_aligned(y, 16) && nb / QB < 0x7FFFFFFF)
        hipLaunchKernelGGL(dequantize_q4_0_lanes, dim3((unsigned)((nb + QB - 1) / QB)), dim3(256), 0, ctx->stream,
                           (const uint8_t *)x, reinterpret_cast<float4_t *>(y), nb);
    else
        hipLaunchKernelGGL(dequantize_q4_0_blocks, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, ctx->stream,
                           (const uint16_t *)x, y, nb);
    GH_LAUNCH_CHECK(ctx, "dequantize_row_q4_0 launch");
}

}  // extern "C"
