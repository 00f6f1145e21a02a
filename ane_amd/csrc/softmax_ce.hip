// softmax_ce.hip — fused classifier softmax + cross-entropy forward/backward on logits [V][S].
//
// Reference op: cross_entropy_loss (training/training_dynamic/cpu_ops.h:68-93; transpose form
// training/stories_cpu_ops.h:71-108) plus the loss-scale pass of training/training_dynamic/train.m:497.
//
// The softmax runs down the STRIDED axis v (columns t are contiguous), so a wave reads whole rows
// with 128-bit loads and every lane owns four columns; no cross-lane traffic is needed until the
// four waves of a workgroup are combined through LDS.
//   pass 1  each workgroup reduces a block of rows to per-column (max, sum exp) partials
//           (online rescaling between 64-row register tiles);
//   combine per column, partials are merged in a fixed order, the target logit is read and the
//           per-column loss term is formed (the mean is taken, by a fixed tree, by one workgroup of pass 2);
//   pass 2  dlogits = (exp(l - M) * (1/L) - onehot) * (1/S) * grad_scale.  Row blocks are visited
//           in the reverse order of pass 1 so the most recently read rows are re-read first
//           (they are the most likely to still sit in the last-level cache).
#include "common.h"
#include "tile.h"

#include <math.h>
#include <algorithm>
#include <type_traits>

namespace {

constexpr int CE_THREADS = 256;
constexpr int CE_WAVES = CE_THREADS / 64;
constexpr int CE_CAP = 16;                       // register tile: 16 steps x 4 waves = 64 rows
constexpr int CE_TILE_ROWS = CE_CAP * CE_WAVES;

template <int VEC>
__device__ __forceinline__ void ld_cols(float (&r)[VEC], const float *p) {
    if constexpr (VEC == 4) {
        v4f t = ld4(p);
        r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
    } else {
        r[0] = *p;
    }
}

template <int VEC>
__device__ __forceinline__ void ld_cols_nt(float (&r)[VEC], const float *p) {
    if constexpr (VEC == 4) {
        v4f t = ld4_nt(p);
        r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
    } else {
        r[0] = __builtin_nontemporal_load(p);
    }
}

// bfloat16 logits (the optional bf16-storage variant): four columns = one 64-bit access; widened to fp32 here,
// so everything below is the same arithmetic for both storage types.
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v2u_any __attribute__((ext_vector_type(2), aligned(2)));     // at any bfloat16 element
__device__ __forceinline__ float bf_widen(unsigned bits16) { return bf_to_f(bits16); }
__device__ __forceinline__ unsigned bf_narrow(float f) { return f_to_bf(f); }      // round to nearest even; NaN stays NaN
template <int VEC>
__device__ __forceinline__ void ld_cols(float (&r)[VEC], const uint16_t *p) {
    if constexpr (VEC == 4) {
        const v2u w = *reinterpret_cast<const v2u_any *>(p);
        r[0] = bf_widen(w[0] & 0xffffu); r[1] = bf_widen(w[0] >> 16);
        r[2] = bf_widen(w[1] & 0xffffu); r[3] = bf_widen(w[1] >> 16);
    } else {
        r[0] = bf_widen(*p);
    }
}
template <int VEC>
__device__ __forceinline__ void ld_cols_nt(float (&r)[VEC], const uint16_t *p) {
    if constexpr (VEC == 4) {
        const v2u w = __builtin_nontemporal_load(reinterpret_cast<const v2u_any *>(p));
        r[0] = bf_widen(w[0] & 0xffffu); r[1] = bf_widen(w[0] >> 16);
        r[2] = bf_widen(w[1] & 0xffffu); r[3] = bf_widen(w[1] >> 16);
    } else {
        r[0] = bf_widen(*p);
    }
}
__device__ __forceinline__ float ld_one(const float *p) { return *p; }
__device__ __forceinline__ float ld_one(const uint16_t *p) { return bf_widen(*p); }
template <int VEC>
__device__ __forceinline__ void st_cols(float *p, const float (&o)[VEC]) {
    if constexpr (VEC == 4) {
        v4f t = {o[0], o[1], o[2], o[3]};
        st4_nt(p, t);
    } else {
        *p = o[0];
    }
}
template <int VEC>
__device__ __forceinline__ void st_cols(uint16_t *p, const float (&o)[VEC]) {
    if constexpr (VEC == 4) {
        v2u w = {bf_narrow(o[0]) | (bf_narrow(o[1]) << 16), bf_narrow(o[2]) | (bf_narrow(o[3]) << 16)};
        __builtin_nontemporal_store(w, reinterpret_cast<v2u_any *>(p));
    } else {
        *p = (uint16_t)bf_narrow(o[0]);
    }
}

// Maximum of a (max, sum exp) pair before it has seen a value above: a finite number, so that what follows needs no case for
// a part that is empty or all -inf (its sum is 0) or holds NaNs only (a maximum does not see them, x - max is one and the
// sum keeps it).  A column with a NaN, with +inf (inf - inf) or of -inf alone (0 / 0) ends as NaNs, loss and gradient, as in
// the sequential loop.
constexpr float NO_MAX = -3.402823466e+38f;

// grid: (row blocks, column strips of 64*VEC)
template <int VEC, typename T>
__global__ __launch_bounds__(CE_THREADS) void ce_partial_kernel(float *__restrict__ pm, float *__restrict__ pl,
                                                                const T *__restrict__ logits, int V, int S,
                                                                int rows_per_block) {
    __shared__ float sm[CE_WAVES][64 * VEC], sl[CE_WAVES][64 * VEC];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = (blockIdx.y * 64 + lane) * VEC;
    const bool col_ok = col < S;
    const int v_lo = blockIdx.x * rows_per_block;
    const int v_hi = min(V, v_lo + rows_per_block);

    float m[VEC], l[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) { m[j] = NO_MAX; l[j] = 0.f; }

    for (int base = v_lo; base < v_hi; base += CE_TILE_ROWS) {
        float x[CE_CAP][VEC];
#pragma unroll
        for (int k = 0; k < CE_CAP; k++) {
            const int v = base + k * CE_WAVES + wave;
            if (v < v_hi && col_ok) ld_cols<VEC>(x[k], logits + (size_t)v * S + col);   // cached: pass 2 re-reads these rows (non-temporal here costs 30 %)
            else {
#pragma unroll
                for (int j = 0; j < VEC; j++) x[k][j] = -INFINITY;
            }
        }
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            float tm = x[0][j];
#pragma unroll
            for (int k = 1; k < CE_CAP; k++) tm = fmaxf(tm, x[k][j]);
            const float nm = fmaxf(m[j], tm);
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < CE_CAP; k++) s += exp_neg_fast(x[k][j] - nm);   // exp(-inf) = 0 for masked rows
            l[j] = l[j] * exp_neg(m[j] - nm) + s;
            m[j] = nm;
        }
    }
#pragma unroll
    for (int j = 0; j < VEC; j++) { sm[wave][lane * VEC + j] = m[j]; sl[wave][lane * VEC + j] = l[j]; }
    __syncthreads();
    if (wave == 0 && col_ok) {
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            float M = sm[0][lane * VEC + j];
#pragma unroll
            for (int w = 1; w < CE_WAVES; w++) M = fmaxf(M, sm[w][lane * VEC + j]);
            float L = 0.f;
#pragma unroll
            for (int w = 0; w < CE_WAVES; w++) L += sl[w][lane * VEC + j] * exp_neg(sm[w][lane * VEC + j] - M);
            pm[(size_t)blockIdx.x * S + col + j] = M;
            pl[(size_t)blockIdx.x * S + col + j] = L;
        }
    }
}

// One workgroup per 16 columns: 64 groups of threads each merge an interleaved subset of the row blocks (few
// rounds of loads per thread, S/16 workgroups in flight), then the 64 partial results are merged by a fixed
// tree.  The merge of two (max, sum) pairs is the online-softmax rescaling.
constexpr int CB_COLS = 16, CB_GROUPS = 1024 / CB_COLS;
// PLAIN: the stand-alone column softmax; there are no targets, and colInv receives the sum itself (that op divides).
template <typename T, bool PLAIN = false>
__global__ __launch_bounds__(1024) void ce_combine_kernel(float *__restrict__ colM, float *__restrict__ colInv,
                                                          float *__restrict__ colLoss, const float *__restrict__ pm,
                                                          const float *__restrict__ pl,
                                                          const T *__restrict__ logits,
                                                          const int32_t *__restrict__ targets, int V, int S,
                                                          int nblk) {
    __shared__ float sm[CB_GROUPS][CB_COLS], sl[CB_GROUPS][CB_COLS];
    const int cl = threadIdx.x % CB_COLS, g = threadIdx.x / CB_COLS;
    const int t = blockIdx.x * CB_COLS + cl;
    float m = NO_MAX, l = 0.f;
    if (t < S)
        for (int r0 = g; r0 < nblk; r0 += CB_GROUPS * 4) {
            float mr[4], lr[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {     // four independent loads in flight
                const int r = r0 + CB_GROUPS * u;
                mr[u] = r < nblk ? pm[(size_t)r * S + t] : NO_MAX;
                lr[u] = r < nblk ? pl[(size_t)r * S + t] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const float nm = fmaxf(m, mr[u]);
                l = l * exp_neg(m - nm) + lr[u] * exp_neg(mr[u] - nm);
                m = nm;
            }
        }
    sm[g][cl] = m;
    sl[g][cl] = l;
    __syncthreads();
    for (int half = CB_GROUPS / 2; half > 0; half >>= 1) {
        if (g < half) {
            const float m0 = sm[g][cl], m1 = sm[g + half][cl];
            const float nm = fmaxf(m0, m1);
            sl[g][cl] = sl[g][cl] * exp_neg(m0 - nm) + sl[g + half][cl] * exp_neg(m1 - nm);
            sm[g][cl] = nm;
        }
        __syncthreads();
    }
    if (g == 0 && t < S) {
        const float M = sm[0][cl];
        colM[t] = M;
        if constexpr (PLAIN) {
            colInv[t] = sl[0][cl];
            return;
        }
        const float inv = 1.0f / sl[0][cl];
        colInv[t] = inv;
        const int tgt = targets[t];
        float loss = 0.f;
        if (tgt >= 0 && tgt < V) {
            const float p = exp_neg(ld_one(logits + (size_t)tgt * S + t) - M) * inv;
            loss = -logf(p + 1e-10f);
        }
        colLoss[t] = loss;
    }
}

template <int VEC, typename T>
__global__ __launch_bounds__(CE_THREADS) void ce_grad_kernel(T *dlogits, const T *logits,
                                                             const float *__restrict__ colM,
                                                             const float *__restrict__ colInv,
                                                             const int32_t *__restrict__ targets, int V, int S,
                                                             int rows_per_block, float invS, float grad_scale,
                                                             float *__restrict__ loss_out,
                                                             const float *__restrict__ colLoss) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        // loss = (sum_t colLoss[t]) / S with a fixed summation tree; one workgroup does it on the side
        __shared__ float red[CE_THREADS];
        float sl = 0.f;
        for (int t = threadIdx.x; t < S; t += CE_THREADS) sl += colLoss[t];
        red[threadIdx.x] = sl;
        __syncthreads();
        for (int off = CE_THREADS / 2; off > 0; off >>= 1) {
            if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
            __syncthreads();
        }
        if (threadIdx.x == 0) *loss_out = red[0] / (float)S;
    }
    const int col = (blockIdx.y * 64 + lane) * VEC;
    if (col >= S) return;
    const int rb = gridDim.x - 1 - blockIdx.x;           // reverse order of pass 1
    const int v_lo = rb * rows_per_block;
    const int v_hi = min(V, v_lo + rows_per_block);
    float M[VEC], inv[VEC], sc[VEC];
    int tgt[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) {
        M[j] = colM[col + j];
        inv[j] = colInv[col + j];
        const int tg = targets[col + j];
        const bool ok = tg >= 0 && tg < V;
        tgt[j] = ok ? tg : -1;
        sc[j] = ok ? invS : 1.0f;      // an out-of-range target leaves the column unscaled (stories_cpu_ops.h:98)
    }
    for (int base = v_lo; base < v_hi; base += CE_TILE_ROWS) {
        float x[CE_CAP][VEC];
#pragma unroll
        for (int k = 0; k < CE_CAP; k++) {
            const int v = base + k * CE_WAVES + wave;
            if (v < v_hi) ld_cols_nt<VEC>(x[k], logits + (size_t)v * S + col);
        }
#pragma unroll
        for (int k = 0; k < CE_CAP; k++) {
            const int v = base + k * CE_WAVES + wave;
            if (v < v_hi) {
                float o[VEC];
#pragma unroll
                for (int j = 0; j < VEC; j++) {
                    float p = exp_neg(x[k][j] - M[j]) * inv[j];
                    if (v == tgt[j]) p -= 1.0f;
                    p = p * sc[j];
                    if (grad_scale != 1.0f) p = p * grad_scale;
                    o[j] = p;
                }
                st_cols<VEC>(dlogits + (size_t)v * S + col, o);
            }
        }
    }
}

// probs = exp(l - M) / L: the second pass of the stand-alone column softmax (training/train_large_ane.m:508-516)
template <int VEC>
__global__ __launch_bounds__(CE_THREADS) void softmax_out_kernel(float *probs, const float *logits,
                                                                 const float *__restrict__ colM,
                                                                 const float *__restrict__ colL, int V, int S,
                                                                 int rows_per_block) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = (blockIdx.y * 64 + lane) * VEC;
    if (col >= S) return;
    const int rb = gridDim.x - 1 - blockIdx.x;
    const int v_lo = rb * rows_per_block;
    const int v_hi = min(V, v_lo + rows_per_block);
    float M[VEC], L[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) { M[j] = colM[col + j]; L[j] = colL[col + j]; }
    for (int v = v_lo + wave; v < v_hi; v += CE_WAVES) {
        float x[VEC], o[VEC];
        ld_cols_nt<VEC>(x, logits + (size_t)v * S + col);
#pragma unroll
        for (int j = 0; j < VEC; j++) o[j] = exp_neg(x[j] - M[j]) / L[j];
        st_cols<VEC>(probs + (size_t)v * S + col, o);
    }
}

// NLL on given probabilities (training/train_large_ane.m:519-530).  The loss is formed first, by one workgroup and
// a fixed tree, so that the gradient pass may overwrite the probabilities in place.
__global__ __launch_bounds__(CE_THREADS) void nll_loss_kernel(float *__restrict__ loss_out, const float *__restrict__ probs,
                                                              const int32_t *__restrict__ targets, int V, int S) {
    __shared__ float red[CE_THREADS];
    float sl = 0.f;
    for (int t = threadIdx.x; t < S; t += CE_THREADS) {
        const int tg = targets[t];
        if (tg >= 0 && tg < V) sl -= logf(probs[(size_t)tg * S + t] + 1e-10f);
    }
    red[threadIdx.x] = sl;
    __syncthreads();
    for (int off = CE_THREADS / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss_out = red[0] / (float)S;
}

// dlogits = (probs - onehot) * (1/S), one 128-bit access per lane; n4 = V*S/4 when VEC = 4
template <int VEC>
__global__ __launch_bounds__(256) void nll_grad_kernel(float *dlogits, const float *probs,
                                                       const int32_t *__restrict__ targets, int V, int S, size_t n,
                                                       float invS) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * VEC;
    if (i >= n) return;
    const int v = (int)(i / (size_t)S), t0 = (int)(i - (size_t)v * S);
    float x[VEC], o[VEC];
    ld_cols_nt<VEC>(x, probs + i);
#pragma unroll
    for (int j = 0; j < VEC; j++) {
        float p = x[j];
        if (targets[t0 + j] == v) p -= 1.0f;
        o[j] = p * invS;
    }
    st_cols<VEC>(dlogits + i, o);
}

// ---- the one-launch form: logits stay on the chip between the two passes ---------------------------------------
// The register files and the LDS of the chip together hold more than the logits of the classifier
// ([151936][256] fp32 = 156 MB; 256 compute units x (512 KB of registers + 160 KB of LDS) = 172 MB), so one launch
// with ONE workgroup of 1024 threads per compute unit can read most rows once: a workgroup owns a block of rows of
// one 64-column strip (256-byte row pieces), keeps its last 16 row steps in registers and the 9 before them in LDS
// (25 of the 38 steps of the Qwen3 vocabulary; all of them for 32000 rows, and for bfloat16 storage, whose rows take
// half the space), and reads only the remainder a second time.  Measured at [151936][256]: 63 us against 84 us for
// the three launches (bfloat16: 40 against 87).  The (max, sum exp) partials of the workgroups of a strip (its members)
// are exchanged through tagged 8-byte slots as in the clustered RMSNorm (norm_cluster.h): one relaxed agent-scope
// atomic {fp32 value, launch tag} per slot, a launch counter per workgroup number, nothing to clear, a bounded
// wait.  A member whose wait for a partner expires recomputes that partner's partial from memory with the same
// operations in the same order (same bits), so every member of a strip normalises with identical column sums.
constexpr int CR_THREADS = 1024;
constexpr int CR_W = 64;                     // columns per strip
constexpr int CR_RPS = CR_THREADS / 16;      // rows per step: 16 lanes x 16 B per row piece
constexpr int CR_NW = CR_THREADS / 64;
constexpr int CR_MAX_SPLIT = 128;            // members per strip
constexpr int CR_MAX_STRIPS = 16;
constexpr int CR_LOSS_SLOT = 2 * CR_W;       // after the 64 maxima and 64 sums
constexpr int CR_STRIDE = 136;               // slots per workgroup number
constexpr int CR_MAX_WG = 512;
constexpr int CR_SUB = 4;                    // rows per lane and online step beyond the register rows
constexpr int CR_MAX_STEPS = 64;             // beyond that most rows would be read twice anyway
constexpr size_t CR_XCH_BYTES = (size_t)CR_MAX_WG * CR_STRIDE * 8 + (size_t)CR_MAX_WG * 4 + 256;

struct CeXch {
    unsigned long long *slots;     // [CR_MAX_WG][CR_STRIDE]
    unsigned *cnt;                 // [CR_MAX_WG] launches completed by each workgroup number
    int *fallbacks;                // workgroups whose bounded wait expired, ever (diagnostic)
};
// Storage of the logits: element type, the register form of a lane's four columns of one row (fp32: 16 bytes;
// bfloat16: two packed words, widened at each use), loads, the store that rounds, and how many row steps a
// workgroup keeps in registers (64 of a lane's 128 in both cases) and in LDS (144 KB in both cases).
struct CrF32 {
    typedef float T;
    typedef v4f Raw;
    static constexpr int K_REG = 16, K_LDS = 9;        // of the largest variant
    static __device__ __forceinline__ Raw ld(const T *p) { return ld4(p); }
    static __device__ __forceinline__ Raw ld_nt(const T *p) { return ld4_nt(p); }
    static __device__ __forceinline__ Raw ninf() { Raw r = {-INFINITY, -INFINITY, -INFINITY, -INFINITY}; return r; }
    static __device__ __forceinline__ float at(const Raw &r, int j) { return r[j]; }
    template <bool NT>
    static __device__ __forceinline__ void st(T *p, const float (&o)[4]) {
        const Raw r = {o[0], o[1], o[2], o[3]};
        if constexpr (NT) st4_nt(p, r); else st4(p, r);
    }
    static __device__ __forceinline__ void forget(Raw &) {}
};
struct CrBf16 {
    typedef uint16_t T;
    typedef v2u Raw;
    static constexpr int K_REG = 32, K_LDS = 18;       // of the largest variant
    static __device__ __forceinline__ Raw ld(const T *p) { return *reinterpret_cast<const v2u_any *>(p); }
    static __device__ __forceinline__ Raw ld_nt(const T *p) { return __builtin_nontemporal_load(reinterpret_cast<const v2u_any *>(p)); }
    static __device__ __forceinline__ Raw ninf() { Raw r = {0xff80ff80u, 0xff80ff80u}; return r; }
    static __device__ __forceinline__ float at(const Raw &r, int j) { return bf_to_f((j & 1) ? r[j >> 1] >> 16 : r[j >> 1] & 0xffffu); }
    template <bool NT>
    static __device__ __forceinline__ void st(T *p, const float (&o)[4]) {
        const Raw r = {f2_to_bf2(o[0], o[1]), f2_to_bf2(o[2], o[3])};
        if constexpr (NT) __builtin_nontemporal_store(r, reinterpret_cast<v2u_any *>(p));
        else *reinterpret_cast<v2u_any *>(p) = r;
    }
    // Tells the compiler nothing about the words' contents from here on, so that the widened copies made for the
    // first pass are dropped instead of being kept alive for the second (they would double the register rows).
    static __device__ __forceinline__ void forget(Raw &r) {
        unsigned a = r[0], b = r[1];
        asm volatile("" : "+v"(a), "+v"(b));
        r[0] = a; r[1] = b;
    }
};
template <typename T>
struct CrGeo {
    const T *logits;
    int V, S, strips, sw, csplit, Rm;      // sw columns per strip, Rm rows per member
};
// The columns of lane lc of a strip (lane_cols in tile.h: the short last group of a row of any length takes its
// neighbour's columns again).  The partials of a strip are kept by slot, four per lane: slot 4*lc + j is column col + j
// and counts once, where j >= dup.
__device__ __forceinline__ LaneCols cr_cols(int strip, int sw, int lc, int S) {
    LaneCols l = lane_cols<4>(strip * sw + lc * 4, S);
    l.ok = l.ok && lc * 4 < sw;
    if (!l.ok) l.col = lane_cols<4>(strip * sw, S).col;      // no columns: reads along with lane 0, stores nothing
    return l;
}
// The rows of member p: R of them from v_lo, in K steps of CR_RPS rows.  A lane has its row of every step but the last,
// and of that one if row0 is below `last`.
// Addresses: cr_at() of a step k >= 0 is inside the tensor for every lane and every member, also one without rows: a lane without a row
// in the last step reads the member's last row, and a step behind the last one is the last again.  So no load of a tile stands
// behind a condition.  (Behind conditions the compiler waits for each load before the next wherever it moves a value between
// registers at their end: five of the eight loads of bfloat16 [32000][200] went one after the other, and a member's
// partial was there 5.6 us after its start for now 4.6, of fp32 [24573][256] 6.8 for 5.3.)
struct CrRows {
    int v_lo, K, last;
    unsigned step, off, off_last;      // bytes: a step, this lane's row and columns of a step and of the last one
};
template <typename T>
__device__ __forceinline__ CrRows cr_rows(const CrGeo<T> &g, int p, int col, int row0) {
    CrRows r;
    const int R = max(0, min(g.V - p * g.Rm, g.Rm));
    r.v_lo = min(p * g.Rm, g.V - 1);
    r.K = (R + CR_RPS - 1) / CR_RPS;
    r.last = R > 0 ? R - (r.K - 1) * CR_RPS : 1;
    r.step = (unsigned)(CR_RPS * g.S) * (unsigned)sizeof(T);
    r.off = (unsigned)(row0 * g.S + col) * (unsigned)sizeof(T);
    r.off_last = (unsigned)(min(row0, r.last - 1) * g.S + col) * (unsigned)sizeof(T);
    return r;
}
template <typename T>
__device__ __forceinline__ T *cr_at(T *first, const CrRows &r, int k) {      // first: row v_lo
    const int kk = max(min(k, r.K - 1), 0);
    return (T *)((char *)first + (size_t)((unsigned)kk * r.step) + (kk >= r.K - 1 ? r.off_last : r.off));
}

// (m, l) <- (m, l) merged with N more values: the online-softmax step
template <int N>
__device__ __forceinline__ void online_update(float &m, float &l, const float (&x)[N]) {
    float tm = x[0];
#pragma unroll
    for (int k = 1; k < N; k++) tm = fmaxf(tm, x[k]);
    const float nm = fmaxf(m, tm);
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < N; k++) s += exp_neg_fast(x[k] - nm);        // exp(-inf) = 0 for masked rows
    l = l * exp_neg(m - nm) + s;
    m = nm;
}
// Sixteen (max, sum) pairs per column, [16][CR_P] in LDS -> their merge, in the quad of threads 4c .. 4c+3 of column c
// (waves 0 to 3): the maximum first, then every sum rescaled to it and added in a fixed order.  A pair without rows is
// (NO_MAX, 0).
constexpr int CR_P = CR_W + 16;              // row pitch: the four threads of a quad read four rows of a column
__device__ __forceinline__ void cr_merge16(const float (*wm)[CR_P], const float (*wl)[CR_P], float &M, float &L) {
    const int c = threadIdx.x >> 2, q = threadIdx.x & 3;
    float mm[CR_NW / 4];
    M = NO_MAX;
#pragma unroll
    for (int i = 0; i < CR_NW / 4; i++) { mm[i] = wm[q + 4 * i][c]; M = fmaxf(M, mm[i]); }
    M = fmaxf(M, lane_xor<1>(M));
    M = fmaxf(M, lane_xor<2>(M));
    L = 0.f;
#pragma unroll
    for (int i = 0; i < CR_NW / 4; i++) L += wl[q + 4 * i][c] * exp_neg(mm[i] - M);
    L += lane_xor<1>(L);
    L += lane_xor<2>(L);
}

// The (max, sum exp) partial of member p of a strip over its rows, for the 64 slots of the strip: valid in the quad of
// threads 4c .. 4c+3 of slot c on return.  Of a member's K row steps the last K_REG are the register rows, the K_LDS
// before them the LDS rows, and the first kL = K - K_REG - K_LDS the rows that are read twice.  A lane folds its rows
// into its running (max, sum) four (eight, cr_reg_sub) at a time, in row order: the rows before the register rows, then the register rows.
// KEEP: this workgroup's own rows; the loads run ahead of the arithmetic (asked(): called when the first ones are on their way).  Every condition on a step is the same for the
// whole workgroup (scalar branches); a lane without a row in the last step reads the member's last row and its value
// is replaced when it is folded, as is that of a step that the member does not have.
// Otherwise nothing is kept: one column and one group of four rows at a time, the same operations on the same values
// in the same order (same bits) in a handful of registers, because the caller's own rows stay live in theirs.
// Register rows of the variants that have no others fold eight at a time: a group costs a maximum, an exponential and a product
// beside its values.
constexpr int cr_reg_sub(int k_reg, int k_lds) { return k_lds == 0 && k_reg % 8 == 0 ? 8 : CR_SUB; }
template <typename ST, int K_REG, int K_LDS, bool KEEP, bool NT, typename Asked>
__device__ __forceinline__ void cr_member_partial(const CrGeo<typename ST::T> &g, int strip, int p, typename ST::Raw (&xr)[K_REG],
                                                  typename ST::Raw (*lrow)[CR_THREADS],
                                                  float (*wm)[CR_P], float (*wl)[CR_P], float &Mout, float &Lout,
                                                  Asked asked) {
    typedef typename ST::Raw Raw;
    constexpr int RSUB = cr_reg_sub(K_REG, K_LDS);
    static_assert(K_REG % RSUB == 0, "the register rows fold in whole groups");
    const int lc = threadIdx.x & 15, row0 = threadIdx.x >> 4, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const LaneCols mine = cr_cols(strip, g.sw, lc, g.S);
    const CrRows r = cr_rows(g, p, mine.col, row0);
    const int K = r.K, kR = max(0, K - K_REG), kL = max(0, kR - K_LDS);
    const int mineK = row0 < r.last ? K : K - 1;                  // steps in which this lane has a row
    const typename ST::T *first = g.logits + (size_t)r.v_lo * g.S;
    const Raw ninf = ST::ninf();
    float m[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; j++) { m[j] = NO_MAX; l[j] = 0.f; }
    if constexpr (KEEP) {
        auto foldg = [&](auto &t) {
            constexpr int N = sizeof(t) / sizeof(t[0]);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float xs[N];
#pragma unroll
                for (int u = 0; u < N; u++) xs[u] = ST::at(t[u], j);
                online_update<N>(m[j], l[j], xs);
                // a column at a time: the four in step take 13 registers more than there are ([151936][256] 73 us for 66)
                asm volatile("" : "+v"(m[j]), "+v"(l[j]));
            }
        };
        // the register rows are asked for first and folded last: they are in flight while the other rows stream
        // through two groups of four.  (Rows that stay on the chip may be read past the cache.)
#pragma unroll
        for (int i = 0; i < K_REG; i++) {
            const typename ST::T *at = cr_at(first, r, kR + i);
            xr[i] = NT ? ST::ld_nt(at) : ST::ld(at);
        }
        if (K_LDS == 0 || kR == 0) asked();
        if (K_LDS > 0 && kR > 0) {
            // (a row step behind the last of these, kR - 1, is that one again, and dropped when it is folded)
            auto loadg = [&](Raw (&t)[CR_SUB], int k0) {
#pragma unroll
                for (int u = 0; u < CR_SUB; u++) {
                    const int k = min(k0 + u, kR - 1);
                    const typename ST::T *at = (const typename ST::T *)((const char *)first + (size_t)((unsigned)k * r.step) + r.off);
                    t[u] = NT && K_LDS > 0 && k0 >= kL ? ST::ld_nt(at) : ST::ld(at);
                }
            };
            auto keepg = [&](const Raw (&t)[CR_SUB], int k0) {
#pragma unroll
                for (int u = 0; u < CR_SUB; u++)
                    if (k0 + u >= kL && k0 + u < kR) lrow[k0 + u - kL][threadIdx.x] = t[u];
            };
            auto tail = [&](Raw (&t)[CR_SUB], int k0) {
                if (k0 + CR_SUB > kR) {
#pragma unroll
                    for (int u = 0; u < CR_SUB; u++)
                        if (k0 + u >= kR) t[u] = ninf;
                }
            };
            Raw ta[CR_SUB], tb[CR_SUB];
            loadg(ta, 0);
            loadg(tb, CR_SUB);
            asked();
            for (int k0 = 0; k0 < kR; k0 += 2 * CR_SUB) {
                keepg(ta, k0);
                tail(ta, k0);
                foldg(ta);
                loadg(ta, k0 + 2 * CR_SUB);
                if (k0 + CR_SUB < kR) {
                    keepg(tb, k0 + CR_SUB);
                    tail(tb, k0 + CR_SUB);
                    foldg(tb);
                }
                loadg(tb, k0 + 3 * CR_SUB);
            }
        }
#pragma unroll
        for (int c = 0; c < K_REG / RSUB; c++) {
            const int k0 = kR + c * RSUB;
            if (k0 < K) {                                         // groups past the last step hold nothing
                Raw t[RSUB];
#pragma unroll
                for (int u = 0; u < RSUB; u++) t[u] = xr[c * RSUB + u];
                if (k0 + RSUB >= K) {
#pragma unroll
                    for (int u = 0; u < RSUB; u++)
                        if (k0 + u >= mineK) t[u] = ninf;
                }
                foldg(t);
            }
        }
#pragma unroll
        for (int i = 0; i < K_REG; i++) ST::forget(xr[i]);
    } else {
        const unsigned step = CR_RPS * g.S, loff = row0 * g.S + mine.col;
#pragma unroll 1
        for (int j = 0; j < 4; j++) {
            float mj = NO_MAX, lj = 0.f;
            auto part = [&](auto sub, int kbeg, int kend) {
                constexpr int N = decltype(sub)::value;
#pragma unroll 1
                for (int k0 = kbeg; k0 < kend; k0 += N) {
                    float xs[N];
#pragma unroll
                    for (int u = 0; u < N; u++) {
                        const int k = k0 + u;
                        xs[u] = k < min(kend, mineK) ? ld_one(first + (size_t)k * step + loff + j) : -INFINITY;
                    }
                    online_update<N>(mj, lj, xs);
                }
            };
            part(std::integral_constant<int, CR_SUB>(), 0, kR);
            part(std::integral_constant<int, RSUB>(), kR, K);
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (q == j) { m[q] = mj; l[q] = lj; }
        }
    }
    // the four row groups of a wave (their maximum, then the rescaled sums), then the sixteen waves
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float M = fmaxf(m[j], lane_xor<16>(m[j]));
        M = fmaxf(M, lane_xor<32>(M));
        float L = l[j] * exp_neg(m[j] - M);
        L += lane_xor<16>(L);
        L += lane_xor<32>(L);
        m[j] = M;
        l[j] = L;
    }
    if (lane < 16) {
#pragma unroll
        for (int j = 0; j < 4; j++) { wm[wave][lc * 4 + j] = m[j]; wl[wave][lc * 4 + j] = l[j]; }
    }
    __syncthreads();
    if (threadIdx.x < 4 * CR_W) cr_merge16(wm, wl, Mout, Lout);
    __syncthreads();
}

// The members' partials, MPG members per thread (pm, pl: member grp * mpg + q of slot c) -> the strip's column maxima
// and the reciprocals of its sums, in fM and fInv (valid after the barrier): first within the sixteen groups, then the
// groups.
template <int MPG>
__device__ __forceinline__ void cr_merge_members(const float (&pm)[MPG], const float (&pl)[MPG], float (*wm)[CR_P],
                                                 float (*wl)[CR_P], float *fM, float *fInv) {
    const int c = threadIdx.x & 63, grp = threadIdx.x >> 6;
    float M = pm[0];
#pragma unroll
    for (int q = 1; q < MPG; q++) M = fmaxf(M, pm[q]);
    float L = 0.f;
#pragma unroll
    for (int q = 0; q < MPG; q++) L += pl[q] * exp_neg(pm[q] - M);      // a member that is absent has sum 0
    wm[grp][c] = M;
    wl[grp][c] = L;
    __syncthreads();
    if (threadIdx.x < 4 * CR_W) {
        cr_merge16(wm, wl, M, L);
        if ((threadIdx.x & 3) == 0) { fM[threadIdx.x >> 2] = M; fInv[threadIdx.x >> 2] = 1.0f / L; }
    }
    __syncthreads();
}

// The target of the column of slot threadIdx.x % 64 of a strip, as it stands (asked for early), and what counts of it: -1 where
// the slot has no column of its own or the target is out of range.
template <typename T>
__device__ __forceinline__ int cr_slot_target(const CrGeo<T> &g, int strip, const int32_t *targets) {
    return targets[cr_cols(strip, g.sw, (threadIdx.x & 63) >> 2, g.S).col + (threadIdx.x & 3)];
}
template <typename T>
__device__ __forceinline__ int cr_own_target(const CrGeo<T> &g, int strip, int tg) {
    const LaneCols mine = cr_cols(strip, g.sw, (threadIdx.x & 63) >> 2, g.S);
    return mine.ok && (int)(threadIdx.x & 3) >= mine.dup && tg < g.V ? tg : -1;
}
template <typename T>
__device__ __forceinline__ float cr_slot_logit(const CrGeo<T> &g, int strip, int tg) {
    if (tg < 0) return 0.f;
    return ld_one(g.logits + (size_t)tg * g.S + cr_cols(strip, g.sw, threadIdx.x >> 2, g.S).col + (threadIdx.x & 3));
}
// Sum over the strip's columns of -log(p[target] + 1e-10), by wave 0 (every lane of it ends with the sum).
__device__ __forceinline__ float cr_strip_loss(int tg, float logit, float M, float inv) {
    const float p = exp_neg(logit - M) * inv;
    return wave_sum_far_first(tg >= 0 ? -logf(p + 1e-10f) : 0.f);
}

// Strips, members and the reciprocal of the strips in one word: with the tensors, the counters and the sizes they are the arguments
// that a wave finds in its registers (14 dwords), so that it waits for no argument before it asks for its rows.
// n * recip >> 16 is n / strips for the workgroup numbers: the excess of the reciprocal, below strips / 2^16, times n < 2^9 stays below 1.
struct CrWord {
    int strips, csplit;
    unsigned recip;
    __device__ __forceinline__ int over_strips(int n) const { return (int)((unsigned)n * recip >> 16); }
};
static_assert(CR_MAX_STRIPS < 32 && CR_MAX_SPLIT < 256 && CR_MAX_WG * CR_MAX_STRIPS <= 1 << 16, "the fields and the reciprocal hold");
static inline unsigned cr_word(int strips, int csplit) {
    return (unsigned)strips | (unsigned)csplit << 5 | (unsigned)(((1 << 16) + strips - 1) / strips) << 13;
}
__device__ __forceinline__ CrWord cr_unpack(unsigned w) { return {(int)(w & 31), (int)(w >> 5 & 255), w >> 13}; }

// One bounded wait for a tagged slot.  false: the tag did not arrive within spin_ticks.
__device__ __forceinline__ bool cr_wait_slot(const unsigned long long *sp, unsigned want, int spin_ticks, float &value) {
    const long long t0 = wall_clock64();
    for (;;) {
        const unsigned long long pk = __hip_atomic_load(sp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((unsigned)(pk >> 32) == want) { value = __uint_as_float((unsigned)pk); return true; }
        if (wall_clock64() - t0 >= (long long)spin_ticks) return false;
        __builtin_amdgcn_s_sleep(2);
    }
}

// grid: strips * csplit workgroups, all resident at once (one per compute unit).  Workgroup b: strip b % strips,
// member b / strips, so that the workgroups that read the pieces of one row are neighbours in time.
// K_REG, K_LDS: row steps kept in registers and in LDS.  The variants for few steps are not there for their registers:
// the code of a step is written out once for each, 60 KB (fp32) and 83 KB (bfloat16) for the largest, and a launch that
// runs through it once per wave waits for instructions: with one row step per workgroup ([1000][256]) a launch took
// 12.8 us, 4.8 of them before its partial was ready.
// MEMBERS: the most a strip may have.  128 take a thread 32 registers more for the slots it fetches, so the variants for them hold
// eight row steps in registers and the others in LDS.
// NT: rows are read and written past the caches where their pieces are whole 128-byte lines; where two strips share
// the lines at their border the caches have to put the pieces together ([151936][200] fp32 82 us past them, 75 with
// them; [151936][256] 62 and 88).
template <typename ST, int K_REG, int K_LDS, bool NT, int MEMBERS = CR_MAX_SPLIT / 2>
__global__ __launch_bounds__(CR_THREADS) void ce_resident_kernel(const typename ST::T *__restrict__ logits,
                                                                 const int32_t *__restrict__ targets, unsigned *cnt, int V,
                                                                 int S, unsigned word, int sw, int Rm,
                                                                 typename ST::T *__restrict__ dlogits, float grad_scale,
                                                                 float invS, float *__restrict__ loss_out,
                                                                 unsigned long long *slots, int *fallbacks, int spin_ticks,
                                                                 int take_nothing) {
    typedef typename ST::Raw Raw;
    constexpr int MPG = MEMBERS / CR_NW;           // members per group of 64 threads (thread = group, slot)
    __shared__ Raw lrow[K_LDS > 0 ? K_LDS : 1][K_LDS > 0 ? CR_THREADS : 1];
    __shared__ float wm[CR_NW][CR_P], wl[CR_NW][CR_P];
    __shared__ float fb[2][CR_W];                  // one member's partial on its way to the threads that hold it
    __shared__ __align__(16) float fM[CR_W], fInv[CR_W];
    __shared__ __align__(16) int tgt[CR_W];        // the slots' targets as they stand
    __shared__ float strip_loss[CR_MAX_STRIPS];
    __shared__ unsigned want[MEMBERS], lead[CR_MAX_STRIPS];      // tags of the members, and of the strips' leaders
    __shared__ int failed[MEMBERS], failed_loss[CR_MAX_STRIPS];
    __shared__ int any_failed, any_failed_loss;
    const int tid = threadIdx.x;
    auto rows_of = [&]() { return (Raw (*)[CR_THREADS])lrow; };
    // Workgroups are dealt to the eight XCDs in turn.  The workgroups that read the pieces of one row run at the
    // same time and, where the split allows, on one XCD, so that each L2 sees whole rows.
    const CrWord cw = cr_unpack(word);
    const int strips = cw.strips, csplit = cw.csplit;
    int me, strip;
    if (csplit % 8 == 0) {
        const int xcd = blockIdx.x % 8, q = blockIdx.x / 8;
        me = cw.over_strips(q);
        strip = q - me * strips;
        me = xcd + 8 * me;
    } else {
        me = cw.over_strips(blockIdx.x);
        strip = blockIdx.x - me * strips;
    }
    const int b = me * strips + strip;           // the workgroup number that owns slots and counter
    const CrGeo<typename ST::T> g = {logits, V, S, strips, sw, csplit, Rm};
    // the launch counters and the strip's targets are asked for ahead of the rows and wanted only after them (relaxed atomic
    // loads: the compiler leaves them where they stand)
    auto count = [&](int i) { return __hip_atomic_load(cnt + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    const unsigned c_mem = count(min(tid, csplit - 1) * strips + strip);
    const unsigned c_lead = count(min(tid, strips - 1));         // member 0 of strip s is workgroup s
    const unsigned c_own = count(b);
    const int my_tgt = cr_slot_target(g, strip, targets);

    // ---- pass 1: this member's rows, kept; its partial published
    Raw xr[K_REG];
    float Mp = NO_MAX, Lp = 0.f;
    unsigned my_tag = 0;
    cr_member_partial<ST, K_REG, K_LDS, true, NT>(g, strip, me, xr, rows_of(), wm, wl, Mp, Lp, [&]() {
        my_tag = __builtin_amdgcn_readfirstlane(c_own) + 1u;
        if (tid < csplit) { want[tid] = c_mem + 1u; failed[tid] = 0; }
        if (tid < strips) { lead[tid] = c_lead + 1u; failed_loss[tid] = 0; }
        if (tid < CR_W) tgt[tid] = my_tgt;
        if (tid == 0) any_failed = any_failed_loss = 0;
    });
    if (tid < 4 * CR_W && (tid & 3) < 2)
        __hip_atomic_store(slots + (size_t)b * CR_STRIDE + (tid & 3) * CR_W + (tid >> 2),
                           ((unsigned long long)my_tag << 32) | __float_as_uint((tid & 3) ? Lp : Mp), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    const int own_tgt = me == 0 && tid < CR_W ? cr_own_target(g, strip, tgt[tid]) : -1;
    const float my_logit = cr_slot_logit(g, strip, own_tgt);        // (in flight while the partners' partials are awaited)
    __syncthreads();
    // ---- every member's partial.  Thread (group, slot) fetches the (max, sum) slots of the group's members for
    // its slot: eight of them (sixteen with 128 members).  The loads of a round go out together, so a round costs one trip
    // to the memory side however many of them are still missing.
    const int mc = tid & 63, mgrp = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mpg = (csplit + CR_NW - 1) / CR_NW;                      // members per group, at most MPG
    float pm[MPG], pl[MPG];
    {
        unsigned long long pk[2 * MPG];
        unsigned tag[MPG];
        // member q of the group; one that is not there: the last member once more
        auto member = [&](int q) { return min(mgrp * mpg + q, csplit - 1); };
        auto there = [&](int q) { return q < mpg && mgrp * mpg + q < csplit; };
#pragma unroll
        for (int q = 0; q < MPG; q++) tag[q] = __builtin_amdgcn_readfirstlane(want[member(q)]);
        for (long long t0 = 0;;) {
#pragma unroll
            for (int f = 0; f < 2 * MPG; f++) {
                const char *from = (const char *)(slots + (size_t)(member(f >> 1) * strips + strip) * CR_STRIDE + (f & 1) * CR_W);
                pk[f] = __hip_atomic_load((const unsigned long long *)(from + (unsigned)mc * 8u), __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
            }
            bool all = true;
#pragma unroll
            for (int f = 0; f < 2 * MPG; f++) all = all & ((unsigned)(pk[f] >> 32) == tag[f >> 1]);
            if (all && !take_nothing) break;
            const long long now = wall_clock64();
            if (t0 == 0) t0 = now;
            if (take_nothing || now - t0 >= (long long)spin_ticks) {       // (test mode: every partner counts as late, whatever its slots hold)
#pragma unroll
                for (int f = 0; f < 2 * MPG; f++)
                    if (there(f >> 1) && (take_nothing || (unsigned)(pk[f] >> 32) != tag[f >> 1])) failed[member(f >> 1)] = 1;
                any_failed = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
#pragma unroll
        for (int q = 0; q < MPG; q++) {
            pm[q] = there(q) ? __uint_as_float((unsigned)pk[2 * q]) : NO_MAX;
            pl[q] = there(q) ? __uint_as_float((unsigned)pk[2 * q + 1]) : 0.f;
        }
    }
    // one member's partial from memory, into the threads that hold it
    auto recompute = [&](int s2, int p, float (&qm)[MPG], float (&ql)[MPG]) {
        float M2 = NO_MAX, L2 = 0.f;
        cr_member_partial<ST, K_REG, K_LDS, false, NT>(g, s2, p, xr, rows_of(), wm, wl, M2, L2, []() {});
        if (tid < 4 * CR_W && (tid & 3) == 0) { fb[0][tid >> 2] = M2; fb[1][tid >> 2] = L2; }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < MPG; q++)
            if (q < mpg && mgrp * mpg + q == p) { qm[q] = fb[0][mc]; ql[q] = fb[1][mc]; }
        __syncthreads();
    };
    __syncthreads();
    if (any_failed) {                                                // the same for every thread: read after the barrier
        if (tid == 0) atomicAdd(fallbacks, 1);
        for (int p = 0; p < csplit; p++)
            if (failed[p]) recompute(strip, p, pm, pl);
    }
    cr_merge_members(pm, pl, wm, wl, fM, fInv);
    // ---- the loss: a strip's leader forms the strip's term; wave 0 of workgroup 0 adds the terms in order, before its
    // rows (behind them its loads would queue after the workgroup's stores, 2 us at the end of the launch)
    if (tid < CR_W && me == 0) {
        const float ls = cr_strip_loss(own_tgt, my_logit, fM[tid], fInv[tid]);
        if (tid == 0)
            __hip_atomic_store(slots + (size_t)b * CR_STRIDE + CR_LOSS_SLOT,
                               ((unsigned long long)my_tag << 32) | __float_as_uint(ls), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        if (strip == 0) {
            float val = ls;
            bool late = false;
            if (tid > 0 && tid < strips)
                late = take_nothing || !cr_wait_slot(slots + (size_t)tid * CR_STRIDE + CR_LOSS_SLOT, lead[tid], spin_ticks, val);
            if (tid < strips) strip_loss[tid] = val;
            if (late) { failed_loss[tid] = 1; any_failed_loss = 1; }
            float total = 0.f;
            for (int s2 = 0; s2 < strips; s2++) total += __shfl(val, s2, 64);
            if (tid == 0) *loss_out = total / (float)S;              // (written again below if a term was late)
        }
    }

    // ---- pass 2: dlogits = (exp(l - M) / L - onehot) / S * grad_scale
    {
        const int lc = tid & 15;
        int row0 = tid >> 4;
        asm volatile("" : "+v"(row0));     // the addresses are formed again here instead of being kept from pass 1
        const LaneCols mine = cr_cols(strip, sw, lc, S);
        const CrRows r = cr_rows(g, me, mine.col, row0);
        const int K = r.K, kR = max(0, K - K_REG), kL = max(0, kR - K_LDS);
        const typename ST::T *src = logits + (size_t)r.v_lo * S;
        typename ST::T *dst = dlogits + (size_t)r.v_lo * S;
        // A value costs the exponential and one product: f is 1/L, 1/S and the scale in one.  The targets, one or two of the rows of a
        // workgroup, are put in by a step that knows it has one (`hot`), with 1/L by itself, so that p - 1 is what it would be.
        // With the comparison, the subtraction and three products at every value bfloat16 [32000][200] wrote its rows in 4.1 us, now in 3.6.
        // With the order of the loads: [32000][200] 14.7 -> 12.4 us, fp32 [151936][256] 65 -> 60.4, [24573][256] 16.3 -> 14.6.
        float M[4], f[4];
        int tk[4];                         // the target's row is this lane's row of step k when tk == 64k
        static_assert(CR_MAX_STEPS <= 64, "a bit for each step");
        unsigned long long hot = 0;        // steps in which a lane of the wave has one
#pragma unroll
        for (int j = 0; j < 4; j++) {
            M[j] = fM[lc * 4 + j];
            const int tg = tgt[lc * 4 + j];
            const bool ok = tg >= 0 && tg < V;
            tk[j] = ok ? tg - r.v_lo - row0 : -1;
            // an out-of-range target leaves the column unscaled (stories_cpu_ops.h:98)
            f[j] = (fInv[lc * 4 + j] * (ok ? invS : 1.0f)) * grad_scale;
            int k = mine.ok && tk[j] >= 0 && tk[j] % CR_RPS == 0 && tk[j] / CR_RPS < K ? tk[j] / CR_RPS : -1;
            while (const unsigned long long some = __builtin_amdgcn_ballot_w64(k >= 0)) {
                const int one = __builtin_amdgcn_readlane(k, __builtin_ctzll(some));
                hot |= 1ull << one;
                if (k == one) k = -1;
            }
        }
        auto emit = [&](int k, const Raw &x) {
            float o[4];
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = exp_neg(ST::at(x, j) - M[j]) * f[j];
            if ((hot >> k) & 1) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (tk[j] == CR_RPS * k) o[j] = ((exp_neg(ST::at(x, j) - M[j]) * fInv[lc * 4 + j] - 1.0f) * invS) * grad_scale;
            }
            if (mine.ok && (k < K - 1 || row0 < r.last))
                ST::template st<NT>((typename ST::T *)((char *)dst + (size_t)((unsigned)k * r.step) + r.off), o);
        };
        // the rows read a second time run up to sixteen ahead of their use, in the registers that the register
        // rows leave as they are written out
        auto loadg = [&](Raw (&t)[CR_SUB], int k0) {
#pragma unroll
            for (int u = 0; u < CR_SUB; u++)
                if (k0 + u < kL) {
                    const typename ST::T *at = (const typename ST::T *)((const char *)src + (size_t)((unsigned)(k0 + u) * r.step) + r.off);
                    t[u] = NT ? ST::ld_nt(at) : ST::ld(at);
                }
        };
        auto emitg = [&](const Raw (&t)[CR_SUB], int k0) {
#pragma unroll
            for (int u = 0; u < CR_SUB; u++)
                if (k0 + u < kL) emit(k0 + u, t[u]);
        };
        Raw t0[CR_SUB], t1[CR_SUB], t2[CR_SUB], t3[CR_SUB];
        if constexpr (K_LDS > 0) loadg(t0, 0);
#pragma unroll
        for (int i = 0; i < K_REG; i++) {
            if (kR + i < K) emit(kR + i, xr[i]);
            __builtin_amdgcn_sched_barrier(0);       // one row at a time: the scheduler would otherwise hold them all
        }
        if constexpr (K_LDS > 0) {
            loadg(t1, CR_SUB);
            loadg(t2, 2 * CR_SUB);
            loadg(t3, 3 * CR_SUB);
#pragma unroll 1
            for (int i = 0; i < kR - kL; i++) emit(kL + i, rows_of()[i][tid]);
            for (int k0 = 0; k0 < kL; k0 += 4 * CR_SUB) {
                emitg(t0, k0);
                loadg(t0, k0 + 4 * CR_SUB);
                emitg(t1, k0 + CR_SUB);
                loadg(t1, k0 + 5 * CR_SUB);
                emitg(t2, k0 + 2 * CR_SUB);
                loadg(t2, k0 + 6 * CR_SUB);
                emitg(t3, k0 + 3 * CR_SUB);
                loadg(t3, k0 + 7 * CR_SUB);
            }
        }
    }

    // a strip's loss term that did not arrive: from memory, the same way
    if (b == 0) {
        __syncthreads();
        if (any_failed_loss) {
            for (int s2 = 1; s2 < strips; s2++) {
                if (failed_loss[s2]) {
                    float qm[MPG], ql[MPG];
#pragma unroll
                    for (int q = 0; q < MPG; q++) { qm[q] = NO_MAX; ql[q] = 0.f; }
                    for (int p = 0; p < csplit; p++) recompute(s2, p, qm, ql);
                    cr_merge_members(qm, ql, wm, wl, fM, fInv);
                    if (tid < CR_W) {
                        const int tg = cr_own_target(g, s2, cr_slot_target(g, s2, targets));
                        const float ls = cr_strip_loss(tg, cr_slot_logit(g, s2, tg), fM[tid], fInv[tid]);
                        if (tid == 0) strip_loss[s2] = ls;
                    }
                    __syncthreads();
                }
            }
            if (tid == 0) {
                float total = 0.f;
                for (int s2 = 0; s2 < strips; s2++) total += strip_loss[s2];
                *loss_out = total / (float)S;
            }
        }
    }
    if (tid == 0) cnt[b] = my_tag;
}

// resident workgroups of the second pass per compute unit (asked of the runtime once per storage type)
template <typename T>
int grad_blocks_per_cu() {
    static int cached = 0;
    if (cached == 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, ce_grad_kernel<4, T>, CE_THREADS, 0) != hipSuccess || n <= 0)
            n = 4;
        cached = n;
    }
    return cached;
}

// Scratch of mi355_softmax_ce_noalloc_dev: the first-pass partials and the three per-column arrays, in a
// file-scope device array, so that the call needs no allocation.  One copy per GPU, held until the process ends.
// In host code the array's name is only a handle for the symbol lookup below; kernels and copies use the address
// that the lookup returns for the current device.
// Behind them, in the same array, lies the exchange area of the one-launch kernel (slots and launch counters, which
// must start at zero: the array is zero-initialised when the code object is loaded, and nothing ever clears it).
constexpr size_t CE_SCRATCH_BYTES = (size_t)2 << 20;
constexpr size_t CE_XCH_AREA = (size_t)1 << 20;
static_assert(CR_XCH_BYTES <= CE_XCH_AREA, "the exchange area must fit behind the partials");
constexpr int CE_MAX_DEVICES = 16;
}   // namespace
static __device__ __align__(256) unsigned char scratch[CE_SCRATCH_BYTES + CE_XCH_AREA];
namespace {
unsigned char *g_scratch_ptr[CE_MAX_DEVICES] = {};

template <typename T>
int ce_run(const char *who, T *dlogits, float *loss_dev, const T *logits, const int32_t *targets, int V, int S,
           float grad_scale, bool no_alloc = false) {
    if (!mi355_ready(who)) return -1;
    if (!dlogits || !loss_dev || !logits || !targets) return mi355_fail("%s: NULL pointer", who);
    if (V <= 0 || S <= 0) return mi355_fail("%s: bad shape V=%d S=%d", who, V, S);
    {
        // The one-launch form: rows of 4 to 1024 columns, split into strips of at most 64, out of place (a member that
        // recomputes a partner's partial reads the partner's logits).  One workgroup per compute unit at most, so that
        // all of them are resident at once.  Measured against the three launches, us: fp32 [1000][256] 9.0 against 12 (with one
        // column per lane), [32000][256] 16.7 against 25.7, [151936][256] 63 against 84, [32000][1000] 73 against 88; bfloat16
        // [32000][200] 13.9 against 30.5, [151936][256] 40 against 87.
        // Not for a single strip of fp32 whose members have more than 14 row steps (V > 57344 in 64 members): its 64
        // workgroups leave three quarters of the chip idle.  The line lies where an earlier one-launch kernel lost ([50000][63]
        // 19.0 against 20.0, [65536][63] 20.8 against 20.3); with the present one 64 members are ahead beyond it still ([65536][63] 17.2 against
        // 20.7, [90000][64] 22.1 and 25.1, [151936][63] 37.5 and 37.7) except for few columns ([120000][33] 27.5 and 25.4, [151936][4] 28.2
        // and 24.8).  (bfloat16, whose three launches convert twice: [151936][63] 28 against 67; two strips: [151936][65] 28 against 74.)
        typedef typename std::conditional<std::is_same<T, float>::value, CrF32, CrBf16>::type ST;
        const int cu = g_ctx.num_cu > 0 ? g_ctx.num_cu : 256;
        const int strips_r = (int)ceil_div((size_t)S, (size_t)CR_W);
        // rows of whole 128-byte lines: strips of 64 columns past the caches; other rows: strips of equal width through them.
        // Tensors that start within a line have all their strips share lines; past the caches [151936][256] fp32 takes
        // 121 us at an odd element against 101 through them, bfloat16 75 against 48.  From a half line on, whose 64 bytes
        // are what the memory moves, past the caches is the faster: 90 against 97 at 64 bytes, [90000][256] 44 against 53.
        const bool lines = ((size_t)S * sizeof(T)) % 128 == 0 && (((uintptr_t)logits | (uintptr_t)dlogits) & 63) == 0;
        const int sw = lines ? CR_W : 4 * (int)ceil_div((size_t)S, 4 * (size_t)strips_r);
        unsigned char *base = (g_ctx.device >= 0 && g_ctx.device < CE_MAX_DEVICES) ? g_scratch_ptr[g_ctx.device] : nullptr;
        if (g_ctx.ce_resident >= 0 && base && S >= 4 && strips_r <= CR_MAX_STRIPS && (const void *)dlogits != (const void *)logits) {
            int csplit = std::min(cu / strips_r, CR_MAX_SPLIT / 2);
            const auto rows = [&]() { return csplit > 0 ? (int)ceil_div((size_t)V, (size_t)csplit) : 0; };
            const auto row_steps = [&]() { return (int)ceil_div((size_t)rows(), (size_t)CR_RPS); };
            if (csplit >= 2 && csplit * strips_r <= CR_MAX_WG && csplit * strips_r <= cu && row_steps() <= CR_MAX_STEPS &&
                !(std::is_same<T, float>::value && strips_r == 1 && row_steps() > 14 && g_ctx.ce_resident == 0)) {
                // Few strips: 64 members each leave compute units idle, and twice as many halve their rows for 1 us and more of
                // exchange.  us, 64 / 128 members: fp32 [28672][64] 11.1 / 12.3, [32000][64] 11.4 / 12.3, [40000][64] 14.0 / 12.7, [28673][123] 14.5 / 15.1,
                // [33000][123] 15.8 / 15.0, [86946][128] 25.4 / 24.3, [151936][128] 39.4 / 35.7; bfloat16 [24000][64] 10.9 / 11.9, [32000][64] 11.5 / 12.3,
                // [50000][100] 16.5 / 15.4, [86946][64] 20.9 / 18.3, [151936][128] 33.9 / 26.0, [202000][33] 45 / 31.  (The lines lie at 8 and 9 steps; at 8, the last
                // that a variant without LDS rows takes, 64 are the quicker by 0.8 where the line is before it.)
                // Three strips, 64 / 80 members (a multiple of 8 keeps a strip's workgroups on their XCD; with
                // 85 [120000][150] takes 39 for 32): bfloat16 from the step on from which 64 hold rows elsewhere than in registers:
                // [50000][150] 17.5 / 20.8, [100000][192] 25.8 / 26.1, [130000][192] 28.5 / 31, [140000][192] 33.6 / 32.1, [151936][130] 38.6 / 37.6, [202000][150]
                // 51 / 45.5; fp32 [64000][150] 24.9 / 28.1, [151936][192] 50.4 / 51.1, left as it is.
                // (fp32 strips that take three launches keep 64 members where one is forced: the form that the line above compares.)
                const int many = std::min(cu / strips_r, CR_MAX_SPLIT) & ~7, steps = row_steps();
                const bool few = sizeof(T) == 2 ? strips_r <= 2 || (strips_r == 3 && steps > ST::K_REG)
                                                : (strips_r == 2 && steps > 8) || (strips_r == 1 && steps <= 14);
                if (many > csplit && few && steps > 7) csplit = many;
                const int Rm = rows(), K = row_steps();
                CeXch xch;
                xch.slots = (unsigned long long *)(base + CE_SCRATCH_BYTES);
                xch.cnt = (unsigned *)(base + CE_SCRATCH_BYTES + (size_t)CR_MAX_WG * CR_STRIDE * 8);
                xch.fallbacks = (int *)(base + CE_SCRATCH_BYTES + (size_t)CR_MAX_WG * CR_STRIDE * 8 + (size_t)CR_MAX_WG * 4);
                auto launch = [&](auto kernel) {
                    const int spin = mi355_exchange_spin_ticks();
                    hipLaunchKernelGGL(kernel, dim3((unsigned)(csplit * strips_r)), dim3(CR_THREADS), 0, g_ctx.stream, logits,
                                       targets, xch.cnt, V, S, cr_word(strips_r, csplit), sw, Rm, dlogits, grad_scale,
                                       1.0f / (float)S, loss_dev, xch.slots, xch.fallbacks, spin < 0 ? 0 : spin,
                                       g_ctx.xch_take_nothing > 0 ? 1 : 0);
                };
                if (csplit > CR_MAX_SPLIT / 2 && K <= 8) {
                    if (lines) launch(ce_resident_kernel<ST, 8, 0, true, CR_MAX_SPLIT>);
                    else launch(ce_resident_kernel<ST, 8, 0, false, CR_MAX_SPLIT>);
                } else if (csplit > CR_MAX_SPLIT / 2) {
                    if (lines) launch(ce_resident_kernel<ST, 8, ST::K_LDS, true, CR_MAX_SPLIT>);
                    else launch(ce_resident_kernel<ST, 8, ST::K_LDS, false, CR_MAX_SPLIT>);
                }
                else if (K <= 4) { if (lines) launch(ce_resident_kernel<ST, 4, 0, true>); else launch(ce_resident_kernel<ST, 4, 0, false>); }
                else if (K <= 8) { if (lines) launch(ce_resident_kernel<ST, 8, 0, true>); else launch(ce_resident_kernel<ST, 8, 0, false>); }
                else if (K <= 16) { if (lines) launch(ce_resident_kernel<ST, 16, 0, true>); else launch(ce_resident_kernel<ST, 16, 0, false>); }
                else if (lines) launch(ce_resident_kernel<ST, ST::K_REG, ST::K_LDS, true>);
                else launch(ce_resident_kernel<ST, ST::K_REG, ST::K_LDS, false>);
                LAUNCH_OK("softmax_ce (one launch)");
                return 0;
            }
        }
    }
    // Rows per workgroup: one to six 64-row register tiles, chosen so that the workgroups of a column strip fill the
    // compute units evenly (at least 1.75 per unit, and the last round of them as full as possible); ties go to
    // the larger block, which leaves fewer partials to merge.  At V = 151936 on 256 units: 320 rows, 475
    // workgroups (87 us for the op; 256 rows and 594 workgroups: 91 us; 384 rows and 396: 97 us).
    int rpb = g_ctx.ce_rows;
    if (rpb <= 0) {
        const int cu = g_ctx.num_cu > 0 ? g_ctx.num_cu : 256;
        double best = -1.0;
        rpb = CE_TILE_ROWS;
        for (int t = 1; t <= 6; t++) {
            const long nb = (long)ceil_div((size_t)V, (size_t)t * CE_TILE_ROWS);
            if (t > 1 && nb * 4 < (long)cu * 7) break;
            const long rounds = (nb + cu - 1) / cu;
            const double score = (double)nb / (double)(rounds * cu) + 0.002 * t;
            if (score > best) { best = score; rpb = t * CE_TILE_ROWS; }
        }
    }
    const int nblk = (int)ceil_div((size_t)V, (size_t)rpb);
    // The second pass has no partials to merge and its own blocks: a multiple of 16 rows between 64 and 384 that
    // fills the resident workgroup slots of the chip in as few rounds as it can (four workgroups fit a compute
    // unit: at V = 151936, 160 rows = 950 workgroups for 1024 slots, 83 us for the op; 144 rows = 1056 workgroups,
    // a second round for 32 of them, 98 us; 320 rows, less than half the slots, 88 us).
    int rpb2 = g_ctx.ce_rows2;
    if (rpb2 <= 0) {
        const long slots = (long)(g_ctx.num_cu > 0 ? g_ctx.num_cu : 256) * grad_blocks_per_cu<T>();
        double best = -1.0;
        rpb2 = CE_TILE_ROWS;
        for (int m = CE_TILE_ROWS / 16; m <= 6 * CE_TILE_ROWS / 16; m++) {
            const long nb = (long)ceil_div((size_t)V, (size_t)m * 16);
            const long rounds = (nb + slots - 1) / slots;
            const double score = (double)nb / (double)(rounds * slots) - 0.05 * (double)(rounds - 1) + 1e-4 * m;
            if (score > best) { best = score; rpb2 = m * 16; }
        }
    }
    const int nblk2 = (int)ceil_div((size_t)V, (size_t)rpb2);
    // Four columns per lane where the matrix is large enough to fill the chip with the quarter of the lanes and a row is
    // wide enough for the 256 columns of a wave: [16384][256] 22.1 us so against 18.8 with one column per lane,
    // [32000][256] 27.0 against 28.8, [32000][500] 50 against 66.
    const bool vec_ok = S % 4 == 0 && S >= 160 && (size_t)V * S >= 6000000;
    const int vec = vec_ok ? 4 : 1;
    const int strips = (int)ceil_div((size_t)S, (size_t)64 * vec);
    if (strips > 65535) return mi355_fail("%s: S too large", who);

    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t part_b = al((size_t)nblk * S * sizeof(float)), col_b = al((size_t)S * sizeof(float));
    // The fixed scratch array where it is large enough (it always is for the single strips above, which therefore can be
    // recorded without a call that sizes the workspace), else the workspace.
    char *ws = (g_ctx.device >= 0 && g_ctx.device < CE_MAX_DEVICES) ? (char *)g_scratch_ptr[g_ctx.device] : nullptr;
    if (no_alloc && !ws) return mi355_fail("%s: the scratch array was not located at init", who);
    if (2 * part_b + 3 * col_b > CE_SCRATCH_BYTES) {
        if (no_alloc)
            return mi355_fail("%s: V=%d S=%d needs %zu bytes of scratch, the fixed scratch holds %zu "
                              "(use mi355_softmax_ce_dev, whose workspace grows)", who, V, S, 2 * part_b + 3 * col_b,
                              CE_SCRATCH_BYTES);
        ws = nullptr;
    }
    if (!ws) ws = (char *)mi355_ws(2 * part_b + 3 * col_b);
    if (!ws) return -1;
    float *pm = (float *)ws, *pl = (float *)(ws + part_b);
    float *colM = (float *)(ws + 2 * part_b), *colInv = (float *)(ws + 2 * part_b + col_b);
    float *colLoss = (float *)(ws + 2 * part_b + 2 * col_b);

    const dim3 grid((unsigned)nblk, (unsigned)strips);
    if (vec_ok) hipLaunchKernelGGL((ce_partial_kernel<4, T>), grid, dim3(CE_THREADS), 0, g_ctx.stream, pm, pl, logits, V, S, rpb);
    else hipLaunchKernelGGL((ce_partial_kernel<1, T>), grid, dim3(CE_THREADS), 0, g_ctx.stream, pm, pl, logits, V, S, rpb);
    LAUNCH_OK("softmax_ce partial");
    hipLaunchKernelGGL(ce_combine_kernel<T>, dim3((unsigned)ceil_div((size_t)S, CB_COLS)), dim3(1024), 0, g_ctx.stream, colM,
                       colInv, colLoss, pm, pl, logits, targets, V, S, nblk);
    LAUNCH_OK("softmax_ce combine");
    const dim3 grid2((unsigned)nblk2, (unsigned)strips);
    if (vec_ok)
        hipLaunchKernelGGL((ce_grad_kernel<4, T>), grid2, dim3(CE_THREADS), 0, g_ctx.stream, dlogits, logits, colM, colInv,
                           targets, V, S, rpb2, 1.0f / (float)S, grad_scale, loss_dev, colLoss);
    else
        hipLaunchKernelGGL((ce_grad_kernel<1, T>), grid2, dim3(CE_THREADS), 0, g_ctx.stream, dlogits, logits, colM, colInv,
                           targets, V, S, rpb2, 1.0f / (float)S, grad_scale, loss_dev, colLoss);
    LAUNCH_OK("softmax_ce grad");
    return 0;
}

}   // namespace

// Called by mi355_init with the device current: finds this device's copy of the scratch array, and asks the
// runtime for the second pass's occupancy now so that the entry point below never has to.
int mi355_ce_setup(void) {
    const int dev = g_ctx.device;
    if (dev < 0 || dev >= CE_MAX_DEVICES) return mi355_fail("init: device index %d beyond %d", dev, CE_MAX_DEVICES);
    unsigned char *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) return mi355_fail("init: hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = ptr;
    (void)grad_blocks_per_cu<float>();
    return 0;
}

int *mi355_ce_fallbacks_dev(void) {
    unsigned char *base = (g_ctx.ready && g_ctx.device >= 0 && g_ctx.device < CE_MAX_DEVICES) ? g_scratch_ptr[g_ctx.device] : nullptr;
    return base ? (int *)(base + CE_SCRATCH_BYTES + (size_t)CR_MAX_WG * CR_STRIDE * 8 + (size_t)CR_MAX_WG * 4) : nullptr;
}

// The same op with its scratch in the fixed device array: no hipMalloc, no hipFree, no workspace growth.
MI355_API int mi355_softmax_ce_noalloc_dev(float *dlogits, float *loss_dev, const float *logits, const int32_t *targets,
                                           int V, int S, float grad_scale) {
    return ce_run<float>("softmax_ce_noalloc", dlogits, loss_dev, logits, targets, V, S, grad_scale, true);
}

MI355_API int mi355_softmax_cols_dev(float *probs, const float *logits, int V, int S) {
    if (!mi355_ready("softmax_cols")) return -1;
    if (!probs || !logits) return mi355_fail("softmax_cols: NULL pointer");
    if (V <= 0 || S <= 0) return mi355_fail("softmax_cols: bad shape V=%d S=%d", V, S);
    const int rpb = 4 * CE_TILE_ROWS;
    const int nblk = (int)ceil_div((size_t)V, (size_t)rpb);
    const bool vec_ok = S % 4 == 0;
    const int vec = vec_ok ? 4 : 1;
    const int strips = (int)ceil_div((size_t)S, (size_t)64 * vec);
    if (strips > 65535) return mi355_fail("softmax_cols: S too large");
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t part_b = al((size_t)nblk * S * sizeof(float)), col_b = al((size_t)S * sizeof(float));
    char *ws = (char *)mi355_ws(2 * part_b + 2 * col_b);
    if (!ws) return -1;
    float *pm = (float *)ws, *pl = (float *)(ws + part_b);
    float *colM = (float *)(ws + 2 * part_b), *colL = (float *)(ws + 2 * part_b + col_b);
    const dim3 grid((unsigned)nblk, (unsigned)strips);
    if (vec_ok) hipLaunchKernelGGL((ce_partial_kernel<4, float>), grid, dim3(CE_THREADS), 0, g_ctx.stream, pm, pl, logits, V, S, rpb);
    else hipLaunchKernelGGL((ce_partial_kernel<1, float>), grid, dim3(CE_THREADS), 0, g_ctx.stream, pm, pl, logits, V, S, rpb);
    LAUNCH_OK("softmax_cols partial");
    hipLaunchKernelGGL((ce_combine_kernel<float, true>), dim3((unsigned)ceil_div((size_t)S, CB_COLS)), dim3(1024), 0,
                       g_ctx.stream, colM, colL, nullptr, pm, pl, logits, nullptr, V, S, nblk);
    LAUNCH_OK("softmax_cols combine");
    if (vec_ok) hipLaunchKernelGGL(softmax_out_kernel<4>, grid, dim3(CE_THREADS), 0, g_ctx.stream, probs, logits, colM, colL, V, S, rpb);
    else hipLaunchKernelGGL(softmax_out_kernel<1>, grid, dim3(CE_THREADS), 0, g_ctx.stream, probs, logits, colM, colL, V, S, rpb);
    LAUNCH_OK("softmax_cols out");
    return 0;
}

MI355_API int mi355_nll_from_probs_dev(float *dlogits, float *loss_dev, const float *probs, const int32_t *targets, int V,
                                       int S) {
    if (!mi355_ready("nll_from_probs")) return -1;
    if (!dlogits || !loss_dev || !probs || !targets) return mi355_fail("nll_from_probs: NULL pointer");
    if (V <= 0 || S <= 0) return mi355_fail("nll_from_probs: bad shape V=%d S=%d", V, S);
    const size_t n = (size_t)V * S;
    hipLaunchKernelGGL(nll_loss_kernel, dim3(1), dim3(CE_THREADS), 0, g_ctx.stream, loss_dev, probs, targets, V, S);
    LAUNCH_OK("nll_from_probs loss");
    const bool vec_ok = S % 4 == 0;
    if (vec_ok)
        hipLaunchKernelGGL(nll_grad_kernel<4>, dim3((unsigned)ceil_div(n / 4, 256)), dim3(256), 0, g_ctx.stream, dlogits,
                           probs, targets, V, S, n, 1.0f / (float)S);
    else
        hipLaunchKernelGGL(nll_grad_kernel<1>, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, g_ctx.stream, dlogits, probs,
                           targets, V, S, n, 1.0f / (float)S);
    LAUNCH_OK("nll_from_probs grad");
    return 0;
}

MI355_API int mi355_softmax_ce_dev(float *dlogits, float *loss_dev, const float *logits, const int32_t *targets, int V,
                                   int S, float grad_scale) {
    return ce_run<float>("softmax_ce", dlogits, loss_dev, logits, targets, V, S, grad_scale);
}

// bfloat16 logits and gradient (bit patterns as uint16_t); the loss and every intermediate stay fp32.
MI355_API int mi355_softmax_ce_bf16_dev(uint16_t *dlogits, float *loss_dev, const uint16_t *logits, const int32_t *targets,
                                        int V, int S, float grad_scale) {
    return ce_run<uint16_t>("softmax_ce_bf16", dlogits, loss_dev, logits, targets, V, S, grad_scale);
}
