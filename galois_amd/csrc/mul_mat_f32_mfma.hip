// f32 (or f16) x f32 batched matmul with M > 1 on the matrix cores in full f32: the attention products of a
// prefill (scores = K^T q over many positions, out = V p), which the reference leaves to cuBLAS sgemm for an f32
// src0 (src/cuda.rs:698-782; the f32 arm of CudaMatMul is todo!() at src/cuda.rs:867-879) and to gemm_ex for an f16
// one (src/cuda.rs:881-992).
//
//   dst[i2][m][n] = sum_k a[(i2 / r2) * a_s2 + n * a_s1 + k * a_s0] * b[(i2 * M + m) * K + k]
//
// v_mfma_f32_32x32x2_f32 multiplies and accumulates in f32, so nothing is rounded that the scalar kernels do not
// round (an f16 a is widened exactly).  a may be contiguous along K (a K^T-style view of a cache) or along N (a V-style
// view).  Any K, N, M: rows past the end are computed from the last row and not stored, k past the end is zero.
//
// What bounds it: at a head's 64 or 128 columns V p has few tiles and a long K, and scores have many tiles and a short K, so
// neither fills the device with 128 x 128 tiles staged through LDS (what this kernel replaces); the operands come from
// the caches either way.
//   - A wave owns 32 rows of b and 64 columns of the result (two accumulators) and fetches its operands itself.  The
//     matrix instruction adds over k in any order as long as both operands agree on it, so in a chunk of 16 k lane (r, h)
//     takes k = 8h .. 8h+7: eight consecutive floats of a row that is contiguous along k, and one element per instruction
//     of a row that is contiguous along n (32 lanes = one contiguous piece).  The next chunk is requested before the
//     current one is multiplied; nothing meets at a barrier.
//   - Scores, and V p where that fills the device: the workgroup's four waves own neighbouring columns and all of K.  SPLIT
//     (V p of few tiles): they own the same 64 columns and every fourth chunk of K, and their sums meet in LDS at the
//     end, in wave order.  Merge and idle waves cost, so a short K or many tiles are better whole (wt_split_pays).
// Measured, us, 128 x 128 tiles against this: V p of 32 heads of 64, 300 rows over 600 keys 111.9 -> 22.4, 700 over 700 139.6 ->
// 43.3, 17 over 517 81.1 -> 9.4; 32 heads of 128, 512 over 512 101.3 -> 33.1; scores of the same 29.1 -> 23.5, 61.5 -> 41.3, 13.6
// -> 5.4, 51.8 -> 35.1.  Products with neither side short gain as much: 512 x 4096 x 4096 743 -> 172 (a contiguous along k), 760 -> 227
// (along n), 2048 x 2048 x 2048 386 -> 179, 400 -> 182 (f16 a 367 -> 174); 16 rows of 4096 x 4096, where this kernel begins, 676 -> 149, 731 ->
// 45.
#include "common.h"

namespace {

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int WM = 32, WN = 64, WK = 16;

struct __attribute__((packed, aligned(4))) f32x8 {
    float v[8];
};
struct __attribute__((packed, aligned(2))) f16x8 {
    _Float16 v[8];
};

__device__ __forceinline__ void wt_load8(float (&d)[8], const float *p) {
    const f32x8 t = *reinterpret_cast<const f32x8 *>(p);
#pragma unroll
    for (int e = 0; e < 8; e++) d[e] = t.v[e];
}
__device__ __forceinline__ void wt_load8(_Float16 (&d)[8], const _Float16 *p) {
    const f16x8 t = *reinterpret_cast<const f16x8 *>(p);
#pragma unroll
    for (int e = 0; e < 8; e++) d[e] = t.v[e];
}

template <typename AT, bool K_CONTIG, bool SPLIT>
__global__ __launch_bounds__(256) void gemm_f32_wave_tiles(const AT *__restrict__ a, const float *__restrict__ b,
                                                            float *__restrict__ dst, int K, int N, int M, int r2, int64_t a_s0,
                                                            int64_t a_s1, int64_t a_s2, int n_tiles) {
    __shared__ float part[SPLIT ? 3 : 1][2][16][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, h = lane >> 5;
    const uint32_t tile = blockIdx.z * gridDim.x + blockIdx.x;  // (a launch holds fewer than 2^32 threads along x)
    const int mt = tile / (uint32_t)n_tiles, nt = tile - (uint32_t)mt * n_tiles;
    if (mt > (M - 1) / WM) return;
    const int m0 = mt * WM, i2 = blockIdx.y;
    const int n0 = nt * (SPLIT ? WN : 4 * WN) + (SPLIT ? 0 : wave * WN);
    if (!SPLIT && n0 >= N) return;
    const AT *ab = a + (int64_t)(i2 / r2) * a_s2;
    const float *brow = b + ((int64_t)i2 * M + min(m0 + r, M - 1)) * K;
    const AT *acol[2];  // K_CONTIG: row n of the tile; otherwise its element of row k = 0
#pragma unroll
    for (int t = 0; t < 2; t++) acol[t] = ab + min(n0 + t * 32 + r, N - 1) * a_s1;

    float16_t acc[2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[t][e] = 0.0f;

    float bv[2][8];
    AT av[2][2][8];
    auto request = [&](int buf, int k0) {  // a whole chunk: k0 + 16 <= K
        const int k = k0 + 8 * h;
        wt_load8(bv[buf], brow + k);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            if (K_CONTIG) {
                wt_load8(av[buf][t], acol[t] + k);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) av[buf][t][e] = acol[t][(int64_t)(k + e) * a_s0];
            }
        }
    };
    auto multiply = [&](int buf) {
#pragma unroll
        for (int e = 0; e < 8; e++)
#pragma unroll
            for (int t = 0; t < 2; t++)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(bv[buf][e], (float)av[buf][t][e], acc[t], 0, 0, 0);
    };
    constexpr int STEP = SPLIT ? 4 * WK : WK;
    int k0 = SPLIT ? wave * WK : 0;
    if (k0 + WK <= K) {
        request(0, k0);
        for (; k0 + STEP + WK <= K; k0 += 2 * STEP) {  // two chunks a turn: the buffers keep their registers
            request(1, k0 + STEP);
            __builtin_amdgcn_sched_barrier(0);
            multiply(0);
            if (k0 + 2 * STEP + WK > K) {
                multiply(1);
                k0 += 2 * STEP;
                goto whole_chunks_done;
            }
            request(0, k0 + 2 * STEP);
            __builtin_amdgcn_sched_barrier(0);
            multiply(1);
        }
        multiply(0);
        k0 += STEP;
    }
whole_chunks_done:
    if (k0 < K) {  // the last, partial chunk: k past the end is zero in both operands and read in neither
        const int k = k0 + 8 * h;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const bool in = k + e < K;
            const int kk = in ? k + e : K - 1;
            bv[0][e] = in ? brow[kk] : 0.0f;
#pragma unroll
            for (int t = 0; t < 2; t++) av[0][t][e] = in ? acol[t][K_CONTIG ? (int64_t)kk : (int64_t)kk * a_s0] : (AT)0.0f;
        }
        multiply(0);
    }
    if (SPLIT) {
        if (wave != 0) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) part[wave - 1][t][e][lane] = acc[t][e];
        }
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int w = 0; w < 3; w++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[t][e] += part[w][t][e][lane];
    }
    // C layout of the 32x32 MFMA (A rows = m, B rows = n): column n = lane % 32, row m = 8*(e/4) + 4*(lane/32) + e%4
    float *db = dst + (int64_t)i2 * M * N;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int n = n0 + t * 32 + r;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int m = m0 + 8 * (e >> 2) + 4 * h + (e & 3);
            if (m < M && n < N) db[(size_t)m * N + n] = acc[t][e];
        }
    }
}

// Whether V p is better off with its K dealt to the four waves of a workgroup: rounds of workgroups times what one costs, a
// quarter of the chunks and a merge worth 32 k against all of them.  rows: row tiles of all slices.  Measured over 4112 sizes (K
// 16 .. 4096, N 33 .. 16000, 16 .. 4096 rows, 1 .. 32 slices), us, split / whole: one slice of 4096 x 4096 at 16 rows 45 / 150, 32 heads of 128,
// 512 rows over 512 keys 33 / 52, 8 slices of 1000 columns, 300 rows over 4096 k 219 / 366; the other way 32 slices, 2048 rows of
// 128 k and 2048 columns 601 / 430 (f16 638 / 450), 4096 rows of 16 k and 16000 columns 156 / 45.
bool wt_split_pays(int64_t K, int64_t N, int64_t rows, int64_t cus) {
    if (K <= WK) return false;
    const int64_t split = (N + WN - 1) / WN * rows, whole = (N + 4 * WN - 1) / (4 * WN) * rows;
    const double rounds = split > cus ? (double)split / (double)cus : 1.0;
    return 0.8 * rounds * ((double)K / 4.0 + 32.0) < (double)((whole + cus - 1) / cus) * (double)(K + 16);
}

}  // namespace

// M > 1 rows of b against a contiguous along K (a_s0 == 1) or along N (a_s1 == 1); false when the grid does not
// fit, in which case nothing was launched.
template <typename AT>
bool gh_mul_mat_f32_mfma(galois_hip_ctx *ctx, const AT *a, const float *b, float *dst, int K, int N, int M, int ne02,
                         int ne12, int64_t a_s0, int64_t a_s1, int64_t a_s2) {
    if (ne12 > 65535 || (a_s0 != 1 && a_s1 != 1)) return false;
    const int64_t m_tiles = ((int64_t)M + WM - 1) / WM, cus = ctx->n_cu > 0 ? ctx->n_cu : 256;
    const bool split = a_s0 != 1 && wt_split_pays(K, N, m_tiles * ne12, cus);
    const int64_t n_tiles = ((int64_t)N + (split ? WN : 4 * WN) - 1) / (split ? WN : 4 * WN), tiles = n_tiles * m_tiles;
    const int64_t x = tiles < (1 << 23) ? tiles : 1 << 23;
    if ((tiles + x - 1) / x > 65535) return false;
    const dim3 grid((unsigned)x, (unsigned)ne12, (unsigned)((tiles + x - 1) / x));
#define WT_LAUNCH(K_, S_)                                                                                                     \
    hipLaunchKernelGGL((gemm_f32_wave_tiles<AT, K_, S_>), grid, dim3(256), 0, ctx->stream, a, b, dst, K, N, M, ne12 / ne02, a_s0, \
                       a_s1, a_s2, (int)n_tiles)
    if (a_s0 == 1) WT_LAUNCH(true, false);
    else if (split) WT_LAUNCH(false, true);
    else WT_LAUNCH(false, false);
#undef WT_LAUNCH
    return true;
}
template bool gh_mul_mat_f32_mfma<float>(galois_hip_ctx *, const float *, const float *, float *, int, int, int, int, int,
                                         int64_t, int64_t, int64_t);
template bool gh_mul_mat_f32_mfma<_Float16>(galois_hip_ctx *, const _Float16 *, const float *, float *, int, int, int, int,
                                            int, int64_t, int64_t, int64_t);
