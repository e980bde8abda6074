// A whole LLaMA decode step -- every layer's products, attention, norms and residuals, and the lm head -- in one launch.
//
// Issued op group by op group a layer is four or five dependent launches; each starts with nothing in flight and ends with a
// chain of round trips during which the memory idles (2.9 us of 4 to 25 each).  Here the workgroups of all stages of
// all layers are laid end to end in one grid:
//     per layer:  q | k | v  ->  attention, a workgroup per (split of the keys, head)  ->  merge of a head's splits
//                 ->  wo + residual  ->  silu(gate) * up  ->  down + residual           then the lm head.
// A workgroup requests everything that does not depend on the stage before it (its weights or cache rows, into
// registers), waits for that stage, and finishes.  Two workgroups are resident per CU, so the weights of the next stage or two
// are on their way while a stage computes.  What bounds it: per stage a wait (a store seen by another XCD, 0.6 us), the
// activations (0.8), their preparation and the dot products (the vector ALU: 10 us a layer of 4096 / 11008 in all), 3 to 4 us;
// and that registers hold 55 MB of a layer's 115 to 180.  Measured, us a layer of 4096 / 11008, 32 heads (four launches / this):
// 2045 f32 keys 52 / 43, 201 f16 keys 42 / 34; of 1024 / 2816, 8 heads, 78 f32 keys 22 / 15.
//
// Why the waits end: a workgroup waits only for workgroups of lower index, and each XCD places the workgroups dealt to it (index
// mod 8) in their order, so the unfinished workgroup of the lowest index runs, or has its place as soon as what holds it ends.
// That is how the dispatcher behaves, no promise of the programming model; and it takes that what else holds places does not
// wait in turn for a place this grid holds: grids that do (gh_order) follow one another where they are of one process.
// Two processes that both send such grids to one device are not ordered.  The waits are bounded for these cases, and for a kernel of
// others that holds an XCD for longer: one that runs out makes the logits NaN and sets the context's status word, and every
// later wait of the launch gives up at once.
//
// Vectors between stages are pairs {f32 value, tag}, stored as 8 bytes with device scope.  The tag names the step and
// the layer, so a reader knows from the element itself whether it is the one it waits for: no producer waits for its
// stores to be acknowledged (0.6 us a stage), nothing is reset between steps.  A reader polls the elements it needs, past the
// caches, but only once the last workgroups of the stage before have set a flag, so that polls do not take the memory
// from the weights; product workgroups set it before their dot products, which take longer than the flag.  (A flag per
// workgroup, all awaited: 2.7 us a stage instead of 1.4, stores to the same line queue up behind one another.)
#include "common.h"
#include "gemv_q4_0_body.h"
#include "attn_decode_body.h"

namespace {

constexpr int DS_THREADS = 512, DS_WAVES = 8, DS_L = 5, DS_D = 128;
constexpr int DS_RW = 6, DS_RO = 4;   // rows per wave of q | k | v, gate | up (pairs: half of them) and the lm head; of wo
constexpr int DS_MAX_LAYERS = 40;     // of one launch (kernel arguments are 4 KB); a deeper model takes several
constexpr int DS_ALL_LAYERS = 250;    // tags of a step: DS_TAGS apart, one per layer
constexpr unsigned DS_TAGS = 256;
constexpr int DS_MAX_SPLITS = 64;
constexpr int DS_FLAGS = 8;           // the last workgroups of a stage set a flag when they are done
constexpr int DS_FLAG = 32;           // dwords from flag to flag: stores to one line queue up behind one another
constexpr int DS_HEADER = 64;         // dwords in front of the flags: [0] the step's tag, [32] the tag of a step that gave up

typedef const __attribute__((address_space(1))) uint8_t *ds_global;

struct ds_layer {
    const uint8_t *wq, *wk, *wv, *wo, *w_gate, *w_up, *w_down;
    const float *attn_norm, *ffn_norm;
    void *kc, *vc;
};

struct ds_args {
    ds_layer layer[DS_MAX_LAYERS];
    const uint8_t *output;
    const float *out_norm;
    float *logits;
    const int32_t *pos;
    unsigned *head;       // workspace header (DS_HEADER dwords), then the flags of the four awaited stages
    unsigned *status;
    uint2 *x, *qkv, *ao, *x1, *h, *rec;
    int32_t first_layer, n_layers, E, F, H, V, L, S;
    int32_t b_qkv, b_attn, b_merge, b_wo, b_ff, b_down, b_layer;  // workgroups of the stages, and of a layer
    int32_t spin_limit;
    uint32_t bias;        // added to what waits wait for: the test hook of the waits
    float eps, freq_scale, theta_scale, scale;
    int64_t key_stride, head_stride;  // of the caches, in elements
};
static_assert(sizeof(ds_args) <= 4096, "kernel arguments");

enum { DS_F_MERGE = 0, DS_F_WO = 1, DS_F_FF = 2, DS_F_DOWN = 3 };

__device__ __forceinline__ unsigned *ds_flags(const ds_args &a, int stage) { return a.head + DS_HEADER + stage * DS_FLAGS * DS_FLAG; }
// The flag of workgroup i of a stage of n, or null.  (The last of a stage start last.)
__device__ __forceinline__ unsigned *ds_flag(const ds_args &a, int stage, int i, int n) {
    const int k = i - (n > DS_FLAGS ? n - DS_FLAGS : 0);
    return k >= 0 ? ds_flags(a, stage) + k * DS_FLAG : nullptr;
}

__device__ __forceinline__ unsigned ds_ld32(const unsigned *p) {
    return __hip_atomic_load(const_cast<unsigned *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint2 ds_ld64(const uint2 *p) {
    const uint64_t v = __hip_atomic_load(reinterpret_cast<uint64_t *>(const_cast<uint2 *>(p)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
}
__device__ __forceinline__ void ds_st64(uint2 *p, float v, unsigned tag) {
    __hip_atomic_store(reinterpret_cast<uint64_t *>(p), (uint64_t)__builtin_bit_cast(uint32_t, v) | (uint64_t)tag << 32, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float ds_f(uint32_t u) { return __builtin_bit_cast(float, u); }

// Bounded waiting of one lane or wave: false when the polls ran out or another workgroup of the step gave up before.
struct ds_wait {
    const ds_args &a;
    unsigned base;
    int left;
    __device__ __forceinline__ ds_wait(const ds_args &a_, unsigned base_) : a(a_), base(base_), left(a_.spin_limit) {}
    __device__ __forceinline__ bool again() {
        --left;
        if ((left & 31) == 0 && ds_ld32(a.head + 32) == base) return false;
        return left > 0;
    }
    __device__ __forceinline__ void gave_up() const {
        __hip_atomic_fetch_or(a.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(a.head + 32, base, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};

// By one wave (the first), behind its stores.
__device__ __forceinline__ void ds_set_flag(unsigned *flag, unsigned tag) {
    if (flag != nullptr && threadIdx.x < 16)  // the whole line's worth of a store
        __hip_atomic_store(flag + threadIdx.x, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Lanes of one wave wait until the flags of a stage of n workgroups have reached tag.
__device__ __forceinline__ bool ds_wait_flags(const ds_args &a, unsigned base, const unsigned *flags, int n, unsigned tag) {
    const int lane = threadIdx.x & 63;
    bool ok = true;
    if (lane < min(n, DS_FLAGS)) {
        ds_wait w(a, base);
        while (ok && (int)(ds_ld32(flags + lane * DS_FLAG) - tag) < 0) {
            if (!w.again()) {
                w.gave_up();
                ok = false;
            }
        }
    }
    return ok;
}

// One lane waits until the N elements p[0 .. N-1] carry the tag; v receives their values.
template <int N>
__device__ __forceinline__ bool ds_wait_elems(const ds_args &a, unsigned base, const uint2 *p, unsigned tag, float (&v)[N]) {
    ds_wait w(a, base);
    for (;;) {
        uint2 t[N];
        bool ok = true;
#pragma unroll
        for (int j = 0; j < N; j++) t[j] = ds_ld64(p + j);
#pragma unroll
        for (int j = 0; j < N; j++) ok &= t[j].y == tag, v[j] = ds_f(t[j].x);
        if (ok) return true;
        if (!w.again()) {
            w.gave_up();
            return false;
        }
    }
}

// The eight activations of task idx = (slot, g) of a tagged vector of n elements, in the nibble order of their weight dword.
// COHERENT: with device scope, for a vector that may still be on its way; otherwise by plain loads first (the 32 CUs of an
// XCD then share one trip past its L2), for one that is usually complete.  An element (8 bytes, aligned) arrives whole;
// one that carries an older tag is requested again, with device scope.
typedef uint32_t ds_u4 __attribute__((ext_vector_type(4)));
template <bool COHERENT>
struct ds_task {
    ds_u4 l0, l1, h0, h1;
    __device__ __forceinline__ void load(const uint2 *x, int n, int idx) {
        const int b = (idx >> 3) * 64 + xprep::group_x_index(idx & 7, 0);
        if (COHERENT) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint2 *>(x), 0, n * 8, 0x00027000);
            constexpr int SC1 = 16;
            l0 = __builtin_amdgcn_raw_buffer_load_b128(r, b * 8, 0, SC1), l1 = __builtin_amdgcn_raw_buffer_load_b128(r, b * 8 + 16, 0, SC1);
            h0 = __builtin_amdgcn_raw_buffer_load_b128(r, b * 8 + 128, 0, SC1), h1 = __builtin_amdgcn_raw_buffer_load_b128(r, b * 8 + 144, 0, SC1);
        } else {
            const ds_u4 *lo = reinterpret_cast<const ds_u4 *>(x + b), *hi = reinterpret_cast<const ds_u4 *>(x + b + 16);
            l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
        }
    }
    __device__ __forceinline__ bool carries(unsigned tag) const {
        return ((l0.y ^ tag) | (l0.w ^ tag) | (l1.y ^ tag) | (l1.w ^ tag) | (h0.y ^ tag) | (h0.w ^ tag) | (h1.y ^ tag) | (h1.w ^ tag)) == 0;
    }
    __device__ __forceinline__ bool take(const ds_args &a, unsigned base, const uint2 *x, int n, int idx, unsigned tag, float (&x8)[8]) {
        bool ok = true;
        if (!carries(tag)) {
            ds_wait w(a, base);
            ds_task<true> again;
            for (;;) {
                asm volatile("" ::: "memory");
                again.load(x, n, idx);
                if (again.carries(tag)) break;
                if (!w.again()) {
                    w.gave_up();
                    ok = false;
                    break;
                }
            }
            l0 = again.l0, l1 = again.l1, h0 = again.h0, h1 = again.h1;
        }
        x8[0] = ds_f(l0.x), x8[1] = ds_f(h0.x), x8[2] = ds_f(l0.z), x8[3] = ds_f(h0.z);
        x8[4] = ds_f(l1.x), x8[5] = ds_f(h1.x), x8[6] = ds_f(l1.z), x8[7] = ds_f(h1.z);
        return ok;
    }
};

// Sums over the 64 lanes of R values at once: every step halves the values a lane carries while there are several.  Lane
// `lane` ends with the total of value `row`; first: whether it is the lowest lane that does.
template <int ROWS>
__device__ __forceinline__ float ds_row_sums(const float (&v)[ROWS], int lane, int &row, bool &first) {
    constexpr int R = ROWS <= 2 ? ROWS : (ROWS <= 4 ? 4 : 8);
    static_assert(ROWS <= 8, "rows of a wave");
    float t[R];
#pragma unroll
    for (int i = 0; i < R; i++) t[i] = i < ROWS ? v[i] : 0.0f;
    row = 0;
    int used = 0;
    const bool b0 = lane & 1, b1 = lane & 2, b4 = lane & 16;
    constexpr int R1 = R >= 2 ? R / 2 : 1, R2 = R >= 4 ? R / 4 : 1;
#pragma unroll
    for (int i = 0; i < R1; i++)
        if (R >= 2) {
            const float keep = b0 ? t[2 * i + 1] : t[2 * i], give = b0 ? t[2 * i] : t[2 * i + 1];
            t[i] = keep + dpp_mov<0xB1>(give);  // quad_perm(1,0,3,2)
        } else {
            t[i] += dpp_mov<0xB1>(t[i]);
        }
    if (R >= 2) row |= b0, used |= 1;
#pragma unroll
    for (int i = 0; i < R2; i++)
        if (R >= 4) {
            const float keep = b1 ? t[2 * i + 1] : t[2 * i], give = b1 ? t[2 * i] : t[2 * i + 1];
            t[i] = keep + dpp_mov<0x4E>(give);  // quad_perm(2,3,0,1)
        } else {
            t[i] += dpp_mov<0x4E>(t[i]);
        }
    if (R >= 4) row |= b1 ? 2 : 0, used |= 2;
#pragma unroll
    for (int i = 0; i < R2; i++) {
        t[i] += dpp_mov<0x124>(t[i]);  // row_ror:4
        t[i] += dpp_mov<0x128>(t[i]);  // row_ror:8
    }
    if (R == 8) {
        const float keep = b4 ? t[R2 - 1] : t[0], give = b4 ? t[0] : t[R2 - 1];
        t[0] = keep + __shfl_xor(give, 16, 64);
        row |= b4 ? 4 : 0, used |= 16;
    } else {
        t[0] += __shfl_xor(t[0], 16, 64);
    }
    t[0] += __shfl_xor(t[0], 32, 64);
    first = (lane & ~used) == 0 && row < ROWS;
    return t[0];
}

// ---------------------------------------------------------------------------------------
// A product workgroup: 8 waves of R rows (of R / 2 pairs of rows for a gate / up pair), rows of up to NCH * 64 slots, all
// of the wave's weights in registers before anything is awaited.  Rows per wave: more of them hold more of what is ahead,
// fewer spread a stage's arithmetic more evenly over the CUs (8 / 8 / 8 / 2 of q | k | v, wo, gate | up and down: 38 us a layer
// with 201 f16 keys, 6 / 4 / 6 / 2: 34, 4 / 2 / 4 / 2: 37); 3 rows of down spill.
// RES: a residual is added.  COH: as ds_task.  EARLY: the flag goes up before the dot products.
// NORM: the vector is normalised and weighted by g while it is prepared: w . (inv * x * g) = inv * (w . (x * g)), so the
// product runs on x * g and every wave adds the squares up beside it.
struct ds_product {
    const uint8_t *W, *W2;   // W2: the up matrix of a pair
    int N, ns, wg;           // rows (of one matrix), slots of a row, workgroup of the stage
    const float *g;          // NORM
    const uint2 *x;          // the vector
    unsigned x_tag;
    const unsigned *wait;    // flags of the stage before, or null
    int n_wait;
    const uint2 *res;        // residual or null
    unsigned res_tag;
    uint2 *out;
    float *plain_out;        // instead of out: the logits
    unsigned out_tag;
    unsigned *flag;          // of this workgroup, or null
};

template <int R, int NCH, int PG, bool DUAL, bool NORM, bool RES, bool COH, bool EARLY>
__device__ __forceinline__ void ds_product_wg(const ds_args &a, unsigned base, const ds_product &d, uint32_t *lds) {
    __shared__ float red[DS_WAVES], rows_out[64];
    __shared__ unsigned failed;
    constexpr int SD = slot_lds<DS_L>::dwords, CD = slot_lds<DS_L>::corr_dwords;
    constexpr int RW = DUAL ? R / 2 : R;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int ns = d.ns, row0 = (d.wg * DS_WAVES + wave) * RW;
    const size_t row_bytes = (size_t)ns * sizeof(q4_slot);

    // ---- the weights, then the norm's weight (rows past N are read from row N - 1 and never stored)
    q4_slot q[NCH][R];
#pragma unroll
    for (int c = 0; c < NCH; c++) {
        const uint32_t off = (uint32_t)min(lane + 64 * c, ns - 1) * (uint32_t)sizeof(q4_slot);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint8_t *W = DUAL && r >= RW ? d.W2 : d.W;
            const int row = min(row0 + (DUAL && r >= RW ? r - RW : r), d.N - 1);
            load_slot(q[c][r], W + (size_t)row * row_bytes + off);
        }
    }
    float2 gw[NORM ? PG : 1][4];
    if (NORM) {
#pragma unroll
        for (int p = 0; p < PG; p++) {
            const int idx = min((int)threadIdx.x + p * DS_THREADS, ns * 8 - 1);
            fetch_task(d.g + (size_t)(idx >> 3) * 64, idx & 7, gw[p]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");

    // ---- the stage before
    bool ok = true;
    // the residual of the rows that wave 0 will store: left by a stage before that one
    float res = 0.0f;
    if (RES && wave == 0) {
        const int i = min(d.wg * (DS_WAVES * RW) + lane, d.N - 1);
        float v[1];
        ok &= ds_wait_elems<1>(a, base, d.res + i, d.res_tag, v);
        res = v[0];
    }
    if (wave == 0 && d.wait != nullptr) ok &= ds_wait_flags(a, base, d.wait, d.n_wait, d.x_tag + a.bias);
    if (threadIdx.x == 0) failed = 0;
    __syncthreads();

    // ---- activations: digit planes to LDS
    uint32_t *const corr = lds + ns * SD;
    float ss = 0.0f;
    ds_task<COH> task[2];  // the next one is on its way while one is prepared
    task[0].load(d.x, ns * 64, min((int)threadIdx.x, ns * 8 - 1));
#pragma unroll
    for (int p = 0; p < PG; p++) {
        const int idx = threadIdx.x + p * DS_THREADS;
        if (p + 1 < PG) task[(p + 1) & 1].load(d.x, ns * 64, min(idx + DS_THREADS, ns * 8 - 1));
        if (idx < ns * 8) {
            const int slot = idx >> 3, g = idx & 7;
            float x8[8];
            ok &= task[p & 1].take(a, base, d.x, ns * 64, idx, d.x_tag, x8);
            if (NORM) {
                const float g8[8] = GH_TASK_X8(gw[p]);
#pragma unroll
                for (int j = 0; j < 8; j++) ss = __builtin_fmaf(x8[j], x8[j], ss), x8[j] *= g8[j];
            }
            prep_store<DS_L>(x8, lds + slot * SD, corr + slot * CD, g, [&](float (&y8)[8]) {
#pragma unroll
                for (int j = 0; j < 8; j++) y8[j] = x8[j];
            });
        }
    }
    if (!ok) failed = 1;
    if (NORM) {
        ss = wave_sum(ss);
        if (lane == 0) red[wave] = ss;
    }
    __syncthreads();
    const bool poisoned = failed != 0;
    if (EARLY && wave == 0) ds_set_flag(d.flag, d.out_tag);

    // ---- the rows
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < NCH; c++) {
        const int sl = lane + 64 * c;
        if (sl < ns) slot_rows<DS_L, R>(q[c], lds + sl * SD, corr + sl * CD, acc);
    }
    float inv = 1.0f;
    if (NORM) {
        float tot = 0.0f;
#pragma unroll
        for (int w = 0; w < DS_WAVES; w++) tot += red[w];
        inv = rsqrtf(tot / (float)(ns * 64) + a.eps);
    }
    int row;  // of the wave's, whose total this lane holds; the lanes that store it are the first of theirs
    bool mine;
    float out;
    if (DUAL) {
        float gate[RW], up[RW];
#pragma unroll
        for (int r = 0; r < RW; r++) gate[r] = acc[r], up[r] = acc[RW + r];
        out = ds_row_sums<RW>(gate, lane, row, mine) * inv;
        const float u = ds_row_sums<RW>(up, lane, row, mine) * inv;
        out = out / (1.0f + expf(-out)) * u;
    } else {
        out = ds_row_sums<R>(acc, lane, row, mine) * inv;
    }
    // ---- one wave stores the workgroup's rows: few stores to a line (they queue up), and the flag right behind them
    if (mine) rows_out[wave * RW + row] = out;
    __syncthreads();
    constexpr int ROWS = DS_WAVES * RW;
    static_assert(ROWS <= 64, "one wave stores a workgroup's rows");
    if (wave == 0) {
        row = d.wg * ROWS + lane;
        if (lane < ROWS && row < d.N) {
            out = rows_out[lane];
            if (RES) out += res;
            if (poisoned) out = __builtin_nanf("");
            if (d.plain_out != nullptr)
                d.plain_out[row] = out;
            else
                ds_st64(d.out + row, out, d.out_tag);
        }
        if (!EARLY && d.flag != nullptr) {
            ds_set_flag(d.flag, d.out_tag);
        }
    }
}

// ---------------------------------------------------------------------------------------
// An attention workgroup: KEYS keys (split s) of head h, a lane holding 16 bytes of a cache row.  Every wave runs the
// softmax of its own keys; the eight meet once, at the end.
template <typename CT> struct ds_elems { static constexpr int n = 16 / sizeof(CT); };
template <typename CT> struct ds_keys { static constexpr int n = 512 / sizeof(CT); };  // 128 f32 or 256 f16 keys
__device__ __forceinline__ void ds_unpack(uint4 r, float (&v)[4]) { v[0] = ds_f(r.x), v[1] = ds_f(r.y), v[2] = ds_f(r.z), v[3] = ds_f(r.w); }
__device__ __forceinline__ void ds_unpack(uint4 r, float (&v)[8]) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; i++) v[2 * i] = f16_bits_to_f32(w[i] & 0xFFFFu), v[2 * i + 1] = f16_bits_to_f32(w[i] >> 16);
}

// A lane's pair of q and, where the new position is (kv), of k and v: all requested at once.
__device__ __forceinline__ bool ds_wait_qkv(const ds_args &a, unsigned base, const uint2 *p, bool kv, unsigned tag, float (&q)[2], float (&k)[2],
                                            float (&v)[2]) {
    ds_wait w(a, base);
    const int E = kv ? a.E : 0;
    for (;;) {
        uint2 t[6];
        bool ok = true;
#pragma unroll
        for (int j = 0; j < 6; j++) t[j] = ds_ld64(p + (j & 1) + (j >> 1) * E);
#pragma unroll
        for (int j = 0; j < 6; j++) ok &= t[j].y == tag;
#pragma unroll
        for (int j = 0; j < 2; j++) q[j] = ds_f(t[j].x), k[j] = ds_f(t[2 + j].x), v[j] = ds_f(t[4 + j].x);
        if (ok) return true;
        if (!w.again()) {
            w.gave_up();
            return false;
        }
    }
}

template <typename CT, int KEYS>
__device__ __forceinline__ void ds_attn_wg(const ds_args &a, unsigned base, unsigned tag, int l_idx, const CT *kc_in, const CT *vc_in,
                                           int h, int s) {
    constexpr int EPL = ds_elems<CT>::n, LPR = DS_D / EPL, RPL = 64 / LPR, KPW = KEYS / DS_WAVES, U = KPW / RPL;
    __shared__ __attribute__((aligned(16))) float qs[DS_D];
    __shared__ __attribute__((aligned(16))) CT kn[DS_D], vn[DS_D];
    __shared__ float ored[DS_WAVES][DS_D];
    __shared__ float mred[DS_WAVES], lred[DS_WAVES];
    __shared__ unsigned failed;
    CT *const kc = const_cast<CT *>(kc_in), *const vc = const_cast<CT *>(vc_in);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int sub = lane / LPR, kl = lane % LPR;
    const int l0 = s * KEYS, l1 = min(a.L, l0 + KEYS), lnew = a.L - 1;
    const bool last = l1 == a.L;   // this workgroup holds the new position
    const int kbase = l0 + wave * KPW + sub;
    const size_t hoff = (size_t)h * (size_t)a.head_stride + (size_t)(kl * EPL);

    uint4 kv[U], vv[U];
#pragma unroll
    for (int u = 0; u < U; u++)
        kv[u] = *reinterpret_cast<const uint4 *>(kc + (size_t)min(kbase + u * RPL, l1 - 1) * (size_t)a.key_stride + hoff);
#pragma unroll
    for (int u = 0; u < U; u++)
        vv[u] = *reinterpret_cast<const uint4 *>(vc + (size_t)min(kbase + u * RPL, l1 - 1) * (size_t)a.key_stride + hoff);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");

    // ---- q (and the new position's k and v): a lane of the first wave rotates one pair (rope.cu:3-28, mode 0)
    if (threadIdx.x == 0) failed = 0;
    if (wave == 0) {
        float sn, cs;
        const float p0 = (float)a.pos[0] * a.freq_scale;
        sincosf(p0 * powf(a.theta_scale, (float)lane), &sn, &cs);
        const uint2 *src = a.qkv + (size_t)h * DS_D + 2 * lane;
        float v[2], k[2] = {0.0f, 0.0f}, w[2] = {0.0f, 0.0f};
        const bool ok = ds_wait_qkv(a, base, src, last, tag + a.bias, v, k, w);
        // the same sequence of roundings as rope_rows: one product, then a fused multiply-add
        qs[2 * lane] = __builtin_fmaf(v[0], cs, -(v[1] * sn));
        qs[2 * lane + 1] = __builtin_fmaf(v[0], sn, v[1] * cs);
        if (last) {
            float k0 = __builtin_fmaf(k[0], cs, -(k[1] * sn)), k1 = __builtin_fmaf(k[0], sn, k[1] * cs);
            asm volatile("" : "+v"(k0), "+v"(k1));  // rounded to f32 before it is rounded to the cache's type
            kn[2 * lane] = (CT)k0, kn[2 * lane + 1] = (CT)k1;
            vn[2 * lane] = (CT)w[0], vn[2 * lane + 1] = (CT)w[1];
            const size_t row = (size_t)lnew * (size_t)a.key_stride + (size_t)h * (size_t)a.head_stride + (size_t)(2 * lane);
            kc[row] = (CT)k0, kc[row + 1] = (CT)k1;
            vc[row] = (CT)w[0], vc[row + 1] = (CT)w[1];
        }
        if (!ok) failed = 1;
    }
    __syncthreads();
    const bool poisoned = failed != 0;
    float qv[EPL];
#pragma unroll
    for (int i = 0; i < EPL; i += 4) {
        const float4 t = *reinterpret_cast<const float4 *>(qs + kl * EPL + i);
        qv[i] = t.x, qv[i + 1] = t.y, qv[i + 2] = t.z, qv[i + 3] = t.w;
    }
    if (last) {  // the new row, which the cache did not hold when it was read; keys past it count for nothing
        const uint4 kr = *reinterpret_cast<const uint4 *>(kn + kl * EPL), vr = *reinterpret_cast<const uint4 *>(vn + kl * EPL);
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int l = kbase + u * RPL;
            if (l >= lnew) kv[u] = kr, vv[u] = l == lnew ? vr : make_uint4(0, 0, 0, 0);
        }
    }

    // ---- scores, and the softmax of this wave's keys
    float sc[U], m = -__builtin_inff();
#pragma unroll
    for (int u = 0; u < U; u++) {
        float k[EPL], t = 0.0f;
        ds_unpack(kv[u], k);
#pragma unroll
        for (int i = 0; i < EPL; i++) t = __builtin_fmaf(k[i], qv[i], t);
        t = at_group_sum<LPR>(t) * a.scale;
        sc[u] = kbase + u * RPL < l1 ? t : -__builtin_inff();
        m = fmaxf(m, sc[u]);
    }
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    const float m_ref = m == -__builtin_inff() ? 0.0f : m;  // a wave without a key
    float den = 0.0f, o[EPL];
#pragma unroll
    for (int i = 0; i < EPL; i++) o[i] = 0.0f;
#pragma unroll
    for (int u = 0; u < U; u++) {
        const float p = expf(sc[u] - m_ref);
        float v[EPL];
        ds_unpack(vv[u], v);
        den += p;
#pragma unroll
        for (int i = 0; i < EPL; i++) o[i] = __builtin_fmaf(p, v[i], o[i]);
    }
#pragma unroll
    for (int off = LPR; off < 64; off <<= 1) {
        den += __shfl_xor(den, off, 64);
#pragma unroll
        for (int i = 0; i < EPL; i++) o[i] += __shfl_xor(o[i], off, 64);
    }
    if (sub == 0) {
#pragma unroll
        for (int i = 0; i < EPL; i += 4) *reinterpret_cast<float4 *>(&ored[wave][kl * EPL + i]) = make_float4(o[i], o[i + 1], o[i + 2], o[i + 3]);
    }
    if (lane == 0) mred[wave] = m, lred[wave] = den;
    __syncthreads();
    const int dd = threadIdx.x;
    if (dd < DS_D) {
        float M = mred[0];
#pragma unroll
        for (int w = 1; w < DS_WAVES; w++) M = fmaxf(M, mred[w]);
        const float mr = M == -__builtin_inff() ? 0.0f : M;
        float num = 0.0f, dn = 0.0f;
#pragma unroll
        for (int w = 0; w < DS_WAVES; w++) {
            const float c = expf(mred[w] - mr);
            num = __builtin_fmaf(c, ored[w][dd], num);
            dn = __builtin_fmaf(c, lred[w], dn);
        }
        if (poisoned) num = __builtin_nanf("");
        if (a.S == 1) {
            ds_st64(a.ao + (size_t)l_idx * a.E + (size_t)h * DS_D + dd, num / dn, tag);
        } else {  // record: maximum, denominator, numerators
            uint2 *rec = a.rec + ((size_t)h * a.S + s) * (DS_D + 2);
            ds_st64(rec + 2 + dd, num, tag);
            if (dd == 0) ds_st64(rec, M, tag), ds_st64(rec + 1, dn, tag);
        }
    }
    if (a.S == 1) {
        ds_set_flag(ds_flag(a, DS_F_MERGE, h, a.H), tag);
    }
}

// The merge of a head's splits: thread (group, d) adds up every fourth split for element d.
__device__ __forceinline__ void ds_merge_wg(const ds_args &a, unsigned base, unsigned tag, int l_idx, int h) {
    constexpr int GROUPS = DS_THREADS / DS_D, B = 4;
    __shared__ float num_s[GROUPS][DS_D], m_s[GROUPS], den_s[GROUPS];
    const int d = threadIdx.x % DS_D, grp = threadIdx.x / DS_D;
    const uint2 *rec = a.rec + (size_t)h * a.S * (DS_D + 2);
    float M = -__builtin_inff(), num = 0.0f, den = 0.0f;
    bool ok = true;
    for (int s0 = grp; s0 < a.S; s0 += GROUPS * B) {
        float mm[B], ll[B], oo[B];
        ds_wait w(a, base);
        for (;;) {
            bool all = true;
            uint2 t[3 * B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const uint2 *r = rec + (size_t)min(s0 + j * GROUPS, a.S - 1) * (DS_D + 2);
                t[3 * j] = ds_ld64(r), t[3 * j + 1] = ds_ld64(r + 1), t[3 * j + 2] = ds_ld64(r + 2 + d);
            }
#pragma unroll
            for (int j = 0; j < B; j++) {
                all &= t[3 * j].y == tag && t[3 * j + 1].y == tag && t[3 * j + 2].y == tag;
                mm[j] = s0 + j * GROUPS < a.S ? ds_f(t[3 * j].x) : -__builtin_inff();
                ll[j] = ds_f(t[3 * j + 1].x), oo[j] = ds_f(t[3 * j + 2].x);
            }
            if (all) break;
            if (!w.again()) {
                w.gave_up();
                ok = false;
                break;
            }
        }
        float mn = M;
#pragma unroll
        for (int j = 0; j < B; j++) mn = fmaxf(mn, mm[j]);
        const float mr = mn == -__builtin_inff() ? 0.0f : mn;
        const float c0 = expf(M - mr);
        num *= c0, den *= c0;
#pragma unroll
        for (int j = 0; j < B; j++)
            if (s0 + j * GROUPS < a.S) {
                const float c = expf(mm[j] - mr);
                num = __builtin_fmaf(c, oo[j], num), den = __builtin_fmaf(c, ll[j], den);
            }
        M = mn;
    }
    if (!ok) num = __builtin_nanf("");
    num_s[grp][d] = num;
    if (d == 0) m_s[grp] = M, den_s[grp] = den;
    __syncthreads();
    if (grp == 0) {
        float m = m_s[0];
#pragma unroll
        for (int i = 1; i < GROUPS; i++) m = fmaxf(m, m_s[i]);
        const float mr = m == -__builtin_inff() ? 0.0f : m;
        num = 0.0f, den = 0.0f;
#pragma unroll
        for (int i = 0; i < GROUPS; i++) {
            const float c = expf(m_s[i] - mr);
            num = __builtin_fmaf(c, num_s[i][d], num), den = __builtin_fmaf(c, den_s[i], den);
        }
        ds_st64(a.ao + (size_t)l_idx * a.E + (size_t)h * DS_D + d, num / den, tag);
    }
    ds_set_flag(ds_flag(a, DS_F_MERGE, h, a.H), tag);
}

// RD: rows per wave of down, whose rows are of up to NCHD * 64 slots.
template <typename CT, int RD, int NCHD>
__global__ __launch_bounds__(DS_THREADS, 4) void decode_step(const ds_args a) {
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    const unsigned base = a.head[0];
    const int E = a.E, F = a.F;
    const int li = min((int)blockIdx.x / a.b_layer, a.n_layers);  // layer of this launch; n_layers: the lm head
    int r = (int)blockIdx.x - li * a.b_layer;
    const int l = a.first_layer + li;
    const unsigned tag = base + (unsigned)l;
    ds_product d;
    d.W2 = nullptr, d.g = nullptr, d.res = nullptr, d.res_tag = tag, d.plain_out = nullptr, d.flag = nullptr, d.out_tag = tag;
    d.x_tag = tag, d.ns = E / 64, d.N = E, d.out = nullptr;
    // what the down projections leave is awaited under the tag of the layer that reads it; the first layer of a launch
    // has nothing to wait for
    d.wait = li == 0 ? nullptr : ds_flags(a, DS_F_DOWN), d.n_wait = a.b_down;
    if (li >= a.n_layers) {  // the lm head
        d.W = a.output, d.N = a.V, d.wg = r, d.g = a.out_norm, d.x = a.x + (size_t)l * E, d.plain_out = a.logits;
        ds_product_wg<DS_RW, 1, 1, false, true, false, true, false>(a, base, d, lds);
        return;
    }
    const ds_layer &y = a.layer[li];
    if (r < a.b_qkv) {
        const int per = a.b_qkv / 3, m = r / per;
        d.W = m == 0 ? y.wq : (m == 1 ? y.wk : y.wv), d.wg = r - m * per, d.g = y.attn_norm, d.x = a.x + (size_t)l * E;
        d.out = a.qkv + (size_t)m * E;
        ds_product_wg<DS_RW, 1, 1, false, true, false, true, false>(a, base, d, lds);
        return;
    }
    r -= a.b_qkv;
    if (r < a.b_attn) {
        ds_attn_wg<CT, ds_keys<CT>::n>(a, base, tag, l, (const CT *)y.kc, (const CT *)y.vc, r % a.H, r / a.H);
        return;
    }
    r -= a.b_attn;
    if (r < a.b_merge) {
        ds_merge_wg(a, base, tag, l, r);
        return;
    }
    r -= a.b_merge;
    if (r < a.b_wo) {
        d.W = y.wo, d.wg = r, d.x = a.ao + (size_t)l * E, d.wait = ds_flags(a, DS_F_MERGE), d.n_wait = a.H;
        d.res = a.x + (size_t)l * E, d.out = a.x1 + (size_t)l * E, d.flag = ds_flag(a, DS_F_WO, r, a.b_wo);
        ds_product_wg<DS_RO, 1, 1, false, false, true, false, true>(a, base, d, lds);
        return;
    }
    r -= a.b_wo;
    if (r < a.b_ff) {
        d.W = y.w_gate, d.W2 = y.w_up, d.N = F, d.wg = r, d.g = y.ffn_norm, d.x = a.x1 + (size_t)l * E;
        d.wait = ds_flags(a, DS_F_WO), d.n_wait = a.b_wo, d.out = a.h + (size_t)l * F, d.flag = ds_flag(a, DS_F_FF, r, a.b_ff);
        ds_product_wg<DS_RW, 1, 1, true, true, false, true, true>(a, base, d, lds);
        return;
    }
    r -= a.b_ff;
    d.W = y.w_down, d.ns = F / 64, d.wg = r, d.x = a.h + (size_t)l * F, d.wait = ds_flags(a, DS_F_FF), d.n_wait = a.b_ff;
    d.res = a.x1 + (size_t)l * E, d.out = a.x + (size_t)(l + 1) * E, d.out_tag = tag + 1, d.flag = ds_flag(a, DS_F_DOWN, r, a.b_down);
    ds_product_wg<RD, NCHD, NCHD, false, false, true, true, true>(a, base, d, lds);
}

// In front of a step: the next tag, the token's row of the embedding as the first layer's x (GetRows::f_q_x_f32,
// src/op.rs:2546-2571).  token < 0: the token and its position are the ones on the device.
__global__ __launch_bounds__(1024) void decode_step_begin(const uint16_t *__restrict__ table, int E, int V, unsigned *head, int32_t *token_dev,
                                                          int32_t *pos_dev, int token, int n_past, uint2 *__restrict__ x) {
    unsigned base = head[0] + DS_TAGS;
    if (base == 0) base = DS_TAGS;  // 0 is what a new workspace holds
    const int t = token >= 0 ? token : token_dev[0];
    __syncthreads();
    if (threadIdx.x == 0) {
        head[0] = base;
        if (token >= 0) token_dev[0] = token, pos_dev[0] = n_past;
    }
    const bool bad = t < 0 || t >= V;
    const uint16_t *row = table + (size_t)(bad ? 0 : t) * (size_t)(E / 32) * 9;
    for (int i = threadIdx.x; i < E; i += 1024) {
        const uint16_t *blk = row + (size_t)(i >> 5) * 9;
        const int j = i & 15;
        const uint32_t qs = blk[1 + (j >> 1)] >> ((j & 1) * 8);
        const int n = (int)((i & 16) ? (qs >> 4) & 15u : qs & 15u);
        float v = (float)(n - 8) * f16_bits_to_f32(blk[0]);
        if (bad) v = __builtin_nanf("");
        x[i] = make_uint2(__builtin_bit_cast(uint32_t, v), base);
    }
}

struct ds_shape {
    int rd, nchd, keys;
    int32_t S_max;
    int64_t x, qkv, ao, x1, h, rec, bytes;  // offsets of the vectors, in pairs
};

// Whether a model's step is one this launch takes, and its shape.
bool ds_plan(const galois_hip_llama_model *m, ds_shape &s) {
    const int64_t E = m->n_embd, F = m->n_ff, H = m->n_head;
    if (E <= 0 || F <= 0 || H <= 0 || m->n_vocab <= 0 || m->n_layer <= 0 || m->n_ctx <= 0) return false;
    if (E != H * DS_D || E > 4096 || F % 64 != 0 || F > 12288 || m->n_layer > DS_ALL_LAYERS || m->n_vocab > (1 << 24)) return false;
    s.keys = m->kv_f16 ? ds_keys<_Float16>::n : ds_keys<float>::n;
    s.nchd = (int)((F / 64 + 63) / 64);
    s.rd = s.nchd == 1 ? 4 : 2;
    const int64_t S = ((int64_t)m->n_ctx + s.keys - 1) / s.keys;
    s.S_max = (int32_t)(S < DS_MAX_SPLITS ? S : DS_MAX_SPLITS);
    const int64_t n = m->n_layer;
    int64_t at = (DS_HEADER + 4 * DS_FLAGS * DS_FLAG) / 2;
    s.x = at, at += (n + 1) * E;
    s.qkv = at, at += 3 * E;
    s.ao = at, at += n * E;
    s.x1 = at, at += n * E;
    s.h = at, at += n * F;
    s.rec = at, at += H * s.S_max * (DS_D + 2);
    s.bytes = at * (int64_t)sizeof(uint2);
    return true;
}

template <typename CT>
hipError_t ds_launch(const ds_args &a, const ds_shape &s, unsigned blocks, size_t lds, hipStream_t stream) {
#define DS_GO(RD_, NCHD_)                                                                                                        \
    do {                                                                                                                         \
        const hipError_t e = hipFuncSetAttribute((const void *)decode_step<CT, RD_, NCHD_>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
        if (e != hipSuccess) return e;                                                                                           \
        hipLaunchKernelGGL((decode_step<CT, RD_, NCHD_>), dim3(blocks), dim3(DS_THREADS), lds, stream, a);                       \
        return hipGetLastError();                                                                                                \
    } while (0)
    if (s.nchd == 1) DS_GO(4, 1);
    else if (s.nchd == 2) DS_GO(2, 2);
    else DS_GO(2, 3);
#undef DS_GO
}

}  // namespace

extern "C" int32_t galois_hip_llama_step_workspace(galois_hip_ctx *ctx, const galois_hip_llama_model *model, int64_t *bytes) {
    GH_REQUIRE_CTX(ctx);
    GH_REQUIRE(ctx, model && bytes, GALOIS_HIP_E_NULL, "llama_step_workspace");
    ds_shape s;
    *bytes = ds_plan(model, s) ? s.bytes : 0;
    return GALOIS_HIP_OK;
}

extern "C" int32_t galois_hip_llama_step(galois_hip_ctx *ctx, const galois_hip_llama_model *m, int32_t token, int32_t n_past) {
    GH_REQUIRE_CTX(ctx);
    GH_REQUIRE(ctx, m && m->tok_embd && m->output && m->out_norm && m->logits && m->token && m->pos && m->layers && m->workspace,
               GALOIS_HIP_E_NULL, "llama_step");
    ds_shape s;
    GH_REQUIRE(ctx, ds_plan(m, s), GALOIS_HIP_E_UNSUPPORTED, "llama_step: heads of 128, n_embd up to 4096, n_ff a multiple of 64 up to 12288, up to 250 layers");
    GH_REQUIRE(ctx, n_past >= 0 && n_past < m->n_ctx && token < m->n_vocab, GALOIS_HIP_E_SHAPE, "llama_step: token below n_vocab, n_past below n_ctx");
    GH_REQUIRE(ctx, m->head_major_n_ctx == 0 || m->head_major_n_ctx > n_past, GALOIS_HIP_E_SHAPE,
               "llama_step: head_major_n_ctx is 0 or the capacity of a [n_head][n_ctx][128] cache, above n_past");
    GH_REQUIRE(ctx, m->workspace_bytes >= s.bytes, GALOIS_HIP_E_SHAPE, "llama_step: workspace of galois_hip_llama_step_workspace bytes");
    GH_REQUIRE(ctx, ctx->qkv_attn_launches == 0, GALOIS_HIP_E_UNSUPPORTED, "llama_step: a form of qkv_attn_decode is asked for");
    GH_REQUIRE(ctx, n_past / s.keys < s.S_max, GALOIS_HIP_E_UNSUPPORTED, "llama_step: at most 64 splits of the keys (of 128 in f32, 256 in f16)");
    GH_REQUIRE(ctx, ctx->dev_status_dev != nullptr, GALOIS_HIP_E_UNSUPPORTED, "llama_step: the context has no status word");
    GH_REQUIRE(ctx, gh_aligned(m->tok_embd, 2) && gh_aligned(m->output, 4) && gh_aligned(m->out_norm, 8) && gh_aligned(m->logits, 4) &&
                        gh_aligned(m->token, 4) && gh_aligned(m->pos, 4) && gh_aligned(m->workspace, 256),
               GALOIS_HIP_E_ALIGN, "llama_step");
    for (int32_t i = 0; i < m->n_layer; i++) {
        const galois_hip_llama_layer &y = m->layers[i];
        GH_REQUIRE(ctx, y.wq && y.wk && y.wv && y.wo && y.w_gate && y.w_up && y.w_down && y.attn_norm && y.ffn_norm && y.k_cache && y.v_cache,
                   GALOIS_HIP_E_NULL, "llama_step: a layer's tensor");
        GH_REQUIRE(ctx, gh_aligned(y.wq, 4) && gh_aligned(y.wk, 4) && gh_aligned(y.wv, 4) && gh_aligned(y.wo, 4) && gh_aligned(y.w_gate, 4) &&
                            gh_aligned(y.w_up, 4) && gh_aligned(y.w_down, 4) && gh_aligned(y.attn_norm, 8) && gh_aligned(y.ffn_norm, 8) &&
                            gh_aligned(y.k_cache, 16) && gh_aligned(y.v_cache, 16),
                   GALOIS_HIP_E_ALIGN, "llama_step: matrices 4-byte, norm weights 8-byte, caches 16-byte aligned");
    }
    GH_BIND(ctx);
    ds_args a;
    memset(&a, 0, sizeof(a));
    const int32_t E = m->n_embd, F = m->n_ff, H = m->n_head;
    uint2 *ws = (uint2 *)m->workspace;
    a.output = (const uint8_t *)m->output, a.out_norm = m->out_norm, a.logits = m->logits, a.pos = m->pos;
    a.head = (unsigned *)m->workspace, a.status = ctx->dev_status_dev;
    a.x = ws + s.x, a.qkv = ws + s.qkv, a.ao = ws + s.ao, a.x1 = ws + s.x1, a.h = ws + s.h, a.rec = ws + s.rec;
    a.E = E, a.F = F, a.H = H, a.V = m->n_vocab, a.L = n_past + 1, a.S = (a.L + s.keys - 1) / s.keys;
    const auto wgs = [](int64_t rows, int rows_per_wave) { return (int32_t)((rows + DS_WAVES * rows_per_wave - 1) / (DS_WAVES * rows_per_wave)); };
    a.b_qkv = 3 * wgs(E, DS_RW), a.b_attn = H * a.S, a.b_merge = a.S > 1 ? H : 0, a.b_wo = wgs(E, DS_RO);
    a.b_ff = wgs(F, DS_RW / 2), a.b_down = wgs(E, s.rd);
    a.b_layer = a.b_qkv + a.b_attn + a.b_merge + a.b_wo + a.b_ff + a.b_down;
    a.spin_limit = ctx->wait_spin_limit, a.bias = (uint32_t)ctx->wait_target_bias;
    a.eps = m->rms_eps, a.freq_scale = m->freq_scale, a.theta_scale = m->theta_scale, a.scale = m->scale;
    a.key_stride = m->head_major_n_ctx ? DS_D : E;
    a.head_stride = m->head_major_n_ctx ? (int64_t)m->head_major_n_ctx * DS_D : DS_D;
    const size_t lds = (size_t)(E > F ? E : F) / 64 * slot_lds<DS_L>::bytes_per_slot;
    gh_order order(ctx);
    if (order.status != GALOIS_HIP_OK) return order.status;
    hipLaunchKernelGGL(decode_step_begin, dim3(1), dim3(1024), 0, ctx->stream, (const uint16_t *)m->tok_embd, E, m->n_vocab, a.head, m->token,
                       m->pos, token, n_past, a.x);
    hipError_t e = hipGetLastError();
    for (int32_t first = 0; first < m->n_layer && e == hipSuccess; first += DS_MAX_LAYERS) {
        const int32_t n = m->n_layer - first < DS_MAX_LAYERS ? m->n_layer - first : DS_MAX_LAYERS;
        for (int32_t i = 0; i < n; i++) {
            const galois_hip_llama_layer &y = m->layers[first + i];
            a.layer[i] = {(const uint8_t *)y.wq, (const uint8_t *)y.wk, (const uint8_t *)y.wv, (const uint8_t *)y.wo, (const uint8_t *)y.w_gate,
                          (const uint8_t *)y.w_up, (const uint8_t *)y.w_down, y.attn_norm, y.ffn_norm, y.k_cache, y.v_cache};
        }
        a.first_layer = first, a.n_layers = n;
        const unsigned blocks = (unsigned)n * (unsigned)a.b_layer + (first + n == m->n_layer ? (unsigned)wgs(a.V, DS_RW) : 0u);
        e = m->kv_f16 ? ds_launch<_Float16>(a, s, blocks, lds, ctx->stream) : ds_launch<float>(a, s, blocks, lds, ctx->stream);
    }
    order.launched();
    return gh_hip(ctx, e, "llama_step launch");
}
