// rope.h — RoPE on interleaved row pairs, for float and for bfloat16 storage.
#pragma once
#include "tile.h"

// One lane = one row pair (2i, 2i+1) of a head x one 16-byte group of columns; heads are counted through the batch, those of Q
// first, then those of K.  Bound by memory.
// The lane of a row's short last group loads the row's last whole group, as LaneCols says, and so takes as long as every other
// lane; with a loop over its columns instead, a load and a store in flight at a time in nearly every wave, Q and K of
// [115][12 x 64][54] took 25.2 us (bfloat16: 31.9), now 13.4 (8.1), and [16][12 x 64][500] in bfloat16 16.5, now 9.2.
// It stores that group where nothing that is read can be overwritten by it; in place (own) it stores only the columns that
// are its own, whose inputs no other lane touches ([115][12 x 64][54]: 14.6 us, bfloat16 12.6).
// The stores are nontemporal, the loads are not, since a cache line at the end of a row is asked for twice: [14][12 x 64][256]
// takes 7.8 us (bfloat16 5.2), with plain stores 9.3 (5.6), with nontemporal loads too 9.6 (6.8); [115][12 x 64][54] 13.4 (8.1),
// 18.0 (8.4), 17.4 (11.9).  Two or four heads in one lane, which share the values of the table, take longer: 8.0 (4.9) and
// 14.1 (10.2) with two.
template <int VEC>
__device__ __forceinline__ void rope_load(float (&r)[VEC], const float *p) { ldv<VEC>(r, p); }
template <int VEC>
__device__ __forceinline__ void rope_load(float (&r)[VEC], const bf16_t *p) { ldb<VEC, false>(r, p); }
template <int VEC>
__device__ __forceinline__ void rope_store(float *p, const float (&r)[VEC]) { stv_nt<VEC>(p, r); }
template <int VEC>
__device__ __forceinline__ void rope_store(bf16_t *p, const float (&r)[VEC]) { stb<VEC>(p, r); }
__device__ __forceinline__ void rope_store_one(float *p, float v) { *p = v; }
__device__ __forceinline__ void rope_store_one(bf16_t *p, float v) { *p = (bf16_t)f_to_bf(v); }

constexpr int ROPE_THREADS = 256;
template <typename T, int VEC>
__global__ __launch_bounds__(ROPE_THREADS) void rope_kernel(T *q_out, T *k_out, const T *q_in, const T *k_in, size_t q_heads,
                                                            unsigned half, int S, unsigned cols,
                                                            const float *__restrict__ cos_t, const float *__restrict__ sin_t,
                                                            float sgn, unsigned total, bool own) {
    const unsigned idx = blockIdx.x * ROPE_THREADS + threadIdx.x;
    if (idx >= total) return;
    const unsigned pair = idx / cols, i = pair % half;
    const LaneCols mine = lane_cols<VEC>((int)((idx - pair * cols) * VEC), S);
    const size_t t = (size_t)i * S + mine.col;
    size_t head = pair / half;
    const T *in = q_in;
    T *out = q_out;
    if (head >= q_heads) { head -= q_heads; in = k_in; out = k_out; }
    in += 2 * ((head * half + i) * S) + mine.col;
    out += 2 * ((head * half + i) * S) + mine.col;
    float a[VEC], b[VEC], c[VEC], sn[VEC];
    rope_load<VEC>(a, in);
    rope_load<VEC>(b, in + S);
    constexpr int TV = VEC < 4 ? VEC : 4;
#pragma unroll
    for (int j = 0; j < VEC; j += TV) {
        float ct[TV], st[TV];
        ldv<TV>(ct, cos_t + t + j);
        ldv<TV>(st, sin_t + t + j);
#pragma unroll
        for (int e = 0; e < TV; e++) { c[j + e] = ct[e]; sn[j + e] = st[e] * sgn; }
    }
    float r0[VEC], r1[VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) {      // forward (sgn = +1): x0*c - x1*s, x0*s + x1*c; backward (-1): x0*c + x1*s, -x0*s + x1*c
        r0[j] = a[j] * c[j] - b[j] * sn[j];
        r1[j] = a[j] * sn[j] + b[j] * c[j];
    }
    if (VEC > 1 && own && mine.dup > 0) {
#pragma unroll
        for (int j = 0; j < VEC; j++)
            if (j >= mine.dup) {
                rope_store_one(out + j, r0[j]);
                rope_store_one(out + S + j, r1[j]);
            }
    } else {
        rope_store<VEC>(out, r0);
        rope_store<VEC>(out + S, r1);
    }
}

static inline bool rope_overlap(const void *a, const void *b, size_t na, size_t nb) {
    return na && nb && (const char *)a < (const char *)b + nb && (const char *)b < (const char *)a + na;
}
// hd even, S, batch >= 1, heads + kv_heads >= 1.  Rows shorter than a group go one column per lane.
template <typename T>
static void launch_rope(T *q_out, T *k_out, const T *q_in, const T *k_in, int heads, int kv_heads, int hd, int S, int batch,
                        const float *cos_dev, const float *sin_dev, int dir) {
    constexpr int WIDE = 16 / (int)sizeof(T);
    const size_t half = hd / 2, q_heads = (size_t)batch * heads, k_heads = (size_t)batch * kv_heads;
    const size_t nq = q_heads * hd * S * sizeof(T), nk = k_heads * hd * S * sizeof(T);
    const bool own = S % WIDE != 0 && (rope_overlap(q_out, q_in, nq, nq) || rope_overlap(q_out, k_in, nq, nk) ||
                                       rope_overlap(k_out, q_in, nk, nq) || rope_overlap(k_out, k_in, nk, nk));
    const size_t cols = S < WIDE ? S : ceil_div((size_t)S, WIDE), total = (q_heads + k_heads) * half * cols;
    const dim3 grid((unsigned)ceil_div(total, ROPE_THREADS)), block(ROPE_THREADS);
    if (S < WIDE)
        hipLaunchKernelGGL((rope_kernel<T, 1>), grid, block, 0, g_ctx.stream, q_out, k_out, q_in, k_in, q_heads, (unsigned)half, S,
                           (unsigned)cols, cos_dev, sin_dev, (float)dir, (unsigned)total, own);
    else
        hipLaunchKernelGGL((rope_kernel<T, WIDE>), grid, block, 0, g_ctx.stream, q_out, k_out, q_in, k_in, q_heads, (unsigned)half,
                           S, (unsigned)cols, cos_dev, sin_dev, (float)dir, (unsigned)total, own);
}
