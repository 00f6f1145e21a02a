// staging.hip — fp32 <-> fp16 staging converts and the attention-gradient finish.
//
// The dynamic loop keeps every activation as fp32 [C,S] on the host and converts to fp16 each time a tensor
// goes onto or comes off an accelerator surface (cvt_f32_f16 / cvt_f16_f32,
// training/training_dynamic/io.h:33-50, used by io_write_fp16 / io_read_fp16 / io_write_fp16_at /
// io_write_dyn / io_read_dyn, io.h:53-96, and the per-kernel packers io.h:160-310).  Every one of those is a
// rectangle copy with a conversion: `rows` runs of `cols` contiguous elements, source and destination each
// with their own row pitch.  The converts here take that rectangle.
//
// After the attention backward kernels the loop reads dQ, dK, dV (fp16, all at the query head count),
// sums the query heads of each KV group for dK and dV, copies dQ, and un-rotates dQ and dK
// (training/training_dynamic/train.m:646-660).  attn_grads_finish does that chain in one pass: each
// lane reads its fp16 (or fp32) inputs once and writes the three fp32 results once.
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int ST_THREADS = 256;
constexpr size_t ST_LANES = (size_t)1 << 31;   // of one launch

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h4_any __attribute__((ext_vector_type(4), aligned(2)));
typedef _Float16 h8_any __attribute__((ext_vector_type(8), aligned(2)));      // at any fp16 element of global memory

// ---- rectangle converts: one lane = 16 bytes of the result (8 fp16 or 4 fp32 elements of one row) ----
// Bound by their bytes.  Every store instruction of a wave writes whole lines: with two 16-byte stores 32 bytes apart per
// lane [49152][256] from fp16 took 16.7 us, with one 14.6 (75 MB: 5.2 TB/s).
// Rows of any length (at least a lane's elements) and pitch, at any element: the last lane of a row takes the row's last
// whole group, some of it its neighbour's too, and stores the same values; a rectangle without gaps is one row.  With one
// element per lane where a row was no multiple of 8 or off a 16-byte boundary: [8192][1001] to fp16 15.6 us (now 11.0),
// [24576][1001] from fp16 63.0 (26.7).  Lanes are numbered in 32 bits (a launch holds no more).
__device__ __forceinline__ size_t last_whole(size_t c, size_t n, size_t cols) { return c + n <= cols ? c : cols - n; }

template <bool FAR>
__global__ __launch_bounds__(ST_THREADS) void cvt_f32_f16_v8(_Float16 *__restrict__ dst, size_t dst_ld,
                                                             const float *__restrict__ src, size_t src_ld,
                                                             unsigned colg, size_t cols, size_t total) {
    const unsigned i = blockIdx.x * ST_THREADS + threadIdx.x;
    if (i >= total) return;
    const unsigned r = i / colg;
    const size_t c = last_whole((size_t)8 * (i - r * colg), 8, cols);
    const float *s = src + r * src_ld + c;
    const v4f a = ld4_nt(s), b = ld4_nt(s + 4);
    h8 o;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        o[j] = (_Float16)a[j];       // round to nearest even, overflow to infinity, subnormals kept
        o[4 + j] = (_Float16)b[j];
    }
    if constexpr (FAR) st16_far(dst + r * dst_ld + c, o);
    else __builtin_nontemporal_store(o, reinterpret_cast<h8_any *>(dst + r * dst_ld + c));
}

template <bool FAR>
__global__ __launch_bounds__(ST_THREADS) void cvt_f16_f32_v4(float *__restrict__ dst, size_t dst_ld,
                                                             const _Float16 *__restrict__ src, size_t src_ld,
                                                             unsigned colg, size_t cols, size_t total) {
    const unsigned i = blockIdx.x * ST_THREADS + threadIdx.x;
    if (i >= total) return;
    const unsigned r = i / colg;
    const size_t c = last_whole((size_t)4 * (i - r * colg), 4, cols);
    const h4 v = __builtin_nontemporal_load(reinterpret_cast<const h4_any *>(src + r * src_ld + c));
    v4f a;
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = (float)v[j];
    float *d = dst + r * dst_ld + c;
    st4_stream(d, a, FAR);
}

__global__ __launch_bounds__(ST_THREADS) void cvt_f32_f16_v1(_Float16 *__restrict__ dst, size_t dst_ld,
                                                             const float *__restrict__ src, size_t src_ld,
                                                             size_t cols, size_t total) {
    const size_t i = (size_t)blockIdx.x * ST_THREADS + threadIdx.x;
    if (i >= total) return;
    const size_t r = i / cols, c = i - r * cols;
    dst[r * dst_ld + c] = (_Float16)src[r * src_ld + c];
}

__global__ __launch_bounds__(ST_THREADS) void cvt_f16_f32_v1(float *__restrict__ dst, size_t dst_ld,
                                                             const _Float16 *__restrict__ src, size_t src_ld,
                                                             size_t cols, size_t total) {
    const size_t i = (size_t)blockIdx.x * ST_THREADS + threadIdx.x;
    if (i >= total) return;
    const size_t r = i / cols, c = i - r * cols;
    dst[r * dst_ld + c] = (float)src[r * src_ld + c];
}

// ---- attention-gradient finish ----
template <typename T, int VEC>
struct Cols {
    static_assert(VEC == 1 || VEC == 4, "rows are read 4 columns at a time");
    typedef T Any __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    typedef T Vec __attribute__((ext_vector_type(4)));
    typedef typename std::conditional<VEC == 4, Vec, T>::type Raw;
    static __device__ __forceinline__ Raw load(const T *p) {
        if constexpr (VEC == 4) return __builtin_nontemporal_load(reinterpret_cast<const Any *>(p));
        else return *p;
    }
    static __device__ __forceinline__ float at(const Raw &r, int j) {
        if constexpr (VEC == 4) return (float)r[j];
        else return (float)r;
    }
};

// table rows are shared by every head and sequence: ordinary (cached) loads
template <int VEC>
__device__ __forceinline__ void load_tab(float (&o)[VEC], const float *p) {
    if constexpr (VEC == 1) {
        o[0] = p[0];
    } else {
#pragma unroll
        for (int q = 0; q < VEC / 4; q++) {
            const v4f v = ld4(p + 4 * q);
#pragma unroll
            for (int j = 0; j < 4; j++) o[4 * q + j] = v[j];
        }
    }
}

template <int VEC, bool FAR>
__device__ __forceinline__ void store_cols(float *p, const float (&o)[VEC]) {
    if constexpr (VEC == 1) {
        p[0] = o[0];
    } else {
#pragma unroll
        for (int q = 0; q < VEC / 4; q++) {
            v4f v = {o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]};
            st4_stream(p + 4 * q, v, FAR);
        }
    }
}

// One lane = one interleaved row pair (2i, 2i+1) of one output head x VEC columns (rows of any length >= VEC: the last
// lane of a row as in the converts, so not in place where S % VEC != 0: a neighbour in another wave could read what this
// lane has rotated; one column per lane there).  [8][2048][1001] fp16 in: 89.4 us with one column per lane, now 45.2.
// Four columns per lane for fp16 too, whose stores are then whole lines: [16][2048][256] 22.4 us (117 MB: 5.2 TB/s)
// against 25.2 with eight, [16][2048][250] 24.6 against 26.9 (48.1 with one).  Pair rows are numbered Q heads first, then K heads, then V heads.
// TABLE: dQ and dK are rotated back.  WAVE: rows are whole waves of columns, so that a wave has one row and what follows of its number
// (three divisions among it) is scalar.  ONE: one query head to a KV head, whose K and V rows read only what they use.
template <typename T, int VEC, bool TABLE, bool ONE, bool WAVE, bool FAR>
__global__ __launch_bounds__(ST_THREADS) void attn_grads_finish_kernel(
    const T *qf, const T *__restrict__ kf, const T *__restrict__ vf, int S, int hd, int heads, int kv_heads, int ratio, int batch,
    unsigned total, const float *__restrict__ cos_t, const float *__restrict__ sin_t, size_t sq, size_t sk, size_t sv, float *dq,
    float *__restrict__ dk, float *__restrict__ dv) {
    typedef Cols<T, VEC> Col;
    typedef typename Col::Raw Raw;
    const unsigned idx = blockIdx.x * ST_THREADS + threadIdx.x;
    if (idx >= total) return;
    const unsigned colg = ((unsigned)S + VEC - 1) / VEC;
    unsigned pr, group;
    if constexpr (WAVE) {
        const unsigned wave = __builtin_amdgcn_readfirstlane(idx >> 6);
        pr = wave / (colg >> 6);
        group = ((wave - pr * (colg >> 6)) << 6) + (threadIdx.x & 63);
    } else {
        pr = idx / colg;
        group = idx - pr * colg;
    }
    const int s = (int)last_whole((size_t)group * VEC, VEC, S);
    const unsigned half = (unsigned)hd >> 1;
    const unsigned q_rows = (unsigned)batch * heads * half, kv_rows = (unsigned)batch * kv_heads * half;

    // Each kind of row asks for all it will read before it uses any: with the table read where the rotation is, and a query head
    // when the one before it had been added, a K row of two heads made three trips to memory one after the other
    // ([16][2048][256] with eight KV heads, fp16, 117 MB: 22.8 us, now 21.4 with the scalar rows).  With one head to a KV head there is no
    // second to ask for, and V rows do without the table (read like the others: [16][2048][256] from fp16 29.1 us, so 26.2;
    // [8][768][197] 7.8 and 6.9; from fp32 36.2 and 33.2, 8.7 and 7.7).
    float r0[VEC], r1[VEC], c[VEC], sn[VEC];
    auto ask_table = [&](int i) {
        load_tab<VEC>(c, cos_t + (size_t)i * S + s);
        load_tab<VEC>(sn, sin_t + (size_t)i * S + s);
    };
    auto turn = [&]() {
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            // inverse rotation, written as the forward one with the sine negated
            const float ns = sn[j] * -1.0f;
            const float x0 = r0[j], x1 = r1[j];
            r0[j] = x0 * c[j] - x1 * ns;
            r1[j] = x0 * ns + x1 * c[j];
        }
    };
    float *out;
    if (pr < q_rows) {
        const unsigned bh = pr / half;               // b*heads + h
        const int i = (int)(pr - bh * half);
        const size_t b = bh / (unsigned)heads, h = bh - b * heads;
        const T *in = qf + b * sq + (h * hd + 2 * i) * (size_t)S + s;
        out = dq + ((size_t)bh * hd + 2 * i) * (size_t)S + s;
        if (TABLE) ask_table(i);
        const Raw a0 = Col::load(in), a1 = Col::load(in + S);
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            r0[j] = Col::at(a0, j);
            r1[j] = Col::at(a1, j);
        }
        if (TABLE) turn();
    } else {
        pr -= q_rows;
        const bool is_k = pr < kv_rows;
        if (!is_k) pr -= kv_rows;
        const unsigned bh = pr / half;               // b*kv_heads + kv
        const int i = (int)(pr - bh * half);
        const size_t b = bh / (unsigned)kv_heads, kv = bh - b * kv_heads, head = (size_t)hd * S;
        const T *in = (is_k ? kf + b * sk : vf + b * sv) + ((kv * ratio) * hd + 2 * i) * (size_t)S + s;
        out = (is_k ? dk : dv) + ((size_t)bh * hd + 2 * i) * (size_t)S + s;
        const bool rotated = TABLE && is_k;
        if (ONE ? rotated : TABLE) ask_table(i);     // (for several heads also for V rows: no branch between the loads)
        auto add = [&](const Raw &x0, const Raw &x1) {
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                r0[j] += Col::at(x0, j);
                r1[j] += Col::at(x1, j);
            }
        };
#pragma unroll
        for (int j = 0; j < VEC; j++) r0[j] = r1[j] = 0.f;
        const Raw a0 = Col::load(in), a1 = Col::load(in + S);
        if constexpr (ONE) {
            add(a0, a1);
        } else {
            const Raw b0 = Col::load(in + head), b1 = Col::load(in + head + S);
            __builtin_amdgcn_sched_barrier(0);       // (the compiler would use the first before it asks for the others)
            add(a0, a1);                             // zero, then += in query-head order (io.h:342-350)
            add(b0, b1);
            for (int r = 2; r < ratio; r++) add(Col::load(in + r * head), Col::load(in + r * head + S));
        }
        if (rotated) turn();
    }
    store_cols<VEC, FAR>(out, r0);
    store_cols<VEC, FAR>(out + S, r1);
}

// Results that go out by st16_far: large, and every row of them whole lines.
bool far_rows(const void *dst, size_t pitch_bytes, size_t row_bytes, size_t rows) {
    return row_bytes * rows >= FAR_BYTES && (((uintptr_t)dst | row_bytes | (rows > 1 ? pitch_bytes : 0)) & 127u) == 0;
}

int cvt_args(const char *who, const void *dst, const void *src, size_t dst_ld, size_t src_ld, size_t rows,
             size_t cols) {
    if (!mi355_ready(who)) return -1;
    if (!dst || !src) return mi355_fail("%s: NULL pointer", who);
    if (rows == 0 || cols == 0) return mi355_fail("%s: empty rectangle rows=%zu cols=%zu", who, rows, cols);
    if (dst_ld < cols || src_ld < cols)
        return mi355_fail("%s: row pitch below the row length (cols=%zu dst_ld=%zu src_ld=%zu)", who, cols, dst_ld,
                          src_ld);
    return 0;
}

}   // namespace

MI355_API int mi355_cvt_f32_f16_dev(uint16_t *dst, size_t dst_ld, const float *src, size_t src_ld, size_t rows,
                                    size_t cols) {
    if (cvt_args("cvt_f32_f16", dst, src, dst_ld, src_ld, rows, cols)) return -1;
    _Float16 *d = reinterpret_cast<_Float16 *>(dst);
    if (dst_ld == cols && src_ld == cols) { cols *= rows; rows = 1; }       // no gaps: one row
    if (cols >= 8) {
        const size_t colg = ceil_div(cols, (size_t)8), total = rows * colg;
        auto kernel = far_rows(d, 2 * dst_ld, 2 * cols, rows) ? cvt_f32_f16_v8<true> : cvt_f32_f16_v8<false>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(total, ST_THREADS)), dim3(ST_THREADS), 0,
                           g_ctx.stream, d, dst_ld, src, src_ld, (unsigned)colg, cols, total);
    } else {
        const size_t total = rows * cols;
        hipLaunchKernelGGL(cvt_f32_f16_v1, dim3((unsigned)ceil_div(total, ST_THREADS)), dim3(ST_THREADS), 0,
                           g_ctx.stream, d, dst_ld, src, src_ld, cols, total);
    }
    LAUNCH_OK("cvt_f32_f16");
    return 0;
}

MI355_API int mi355_cvt_f16_f32_dev(float *dst, size_t dst_ld, const uint16_t *src, size_t src_ld, size_t rows,
                                    size_t cols) {
    if (cvt_args("cvt_f16_f32", dst, src, dst_ld, src_ld, rows, cols)) return -1;
    const _Float16 *s = reinterpret_cast<const _Float16 *>(src);
    if (dst_ld == cols && src_ld == cols) { cols *= rows; rows = 1; }       // no gaps: one row
    // (pieces of what one launch can number, for rectangles of more than 8 G elements)
    for (size_t c0 = 0; c0 < cols; c0 += 4 * ST_LANES) {
        const size_t n = std::min(cols - c0, 4 * ST_LANES), colg = n >= 4 ? ceil_div(n, (size_t)4) : n;
        const size_t per = ST_LANES / colg;
        for (size_t r0 = 0; r0 < rows; r0 += per) {
            const size_t total = std::min(rows - r0, per) * colg;
            const dim3 grid((unsigned)ceil_div(total, ST_THREADS));
            float *d = dst + r0 * dst_ld + c0;
            const _Float16 *from = s + r0 * src_ld + c0;
            auto kernel = far_rows(d, 4 * dst_ld, 4 * n, total / colg) ? cvt_f16_f32_v4<true> : cvt_f16_f32_v4<false>;
            if (n >= 4)
                hipLaunchKernelGGL(kernel, grid, dim3(ST_THREADS), 0, g_ctx.stream, d, dst_ld, from, src_ld,
                                   (unsigned)colg, n, total);
            else
                hipLaunchKernelGGL(cvt_f16_f32_v1, grid, dim3(ST_THREADS), 0, g_ctx.stream, d, dst_ld, from, src_ld, n, total);
        }
    }
    LAUNCH_OK("cvt_f16_f32");
    return 0;
}

MI355_API int mi355_attn_grads_finish_dev(float *dq, float *dk, float *dv, const void *dq_full, const void *dk_full,
                                          const void *dv_full, int in_f16, size_t q_stride, size_t k_stride,
                                          size_t v_stride, int heads, int kv_heads, int hd, int S, int batch,
                                          const float *cos_dev, const float *sin_dev) {
    if (!mi355_ready("attn_grads_finish")) return -1;
    if (!dq || !dk || !dv || !dq_full || !dk_full || !dv_full) return mi355_fail("attn_grads_finish: NULL pointer");
    if ((cos_dev == nullptr) != (sin_dev == nullptr))
        return mi355_fail("attn_grads_finish: pass both rotation tables or neither");
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || hd <= 0 || (hd & 1) || S <= 0 || batch <= 0)
        return mi355_fail("attn_grads_finish: bad shape heads=%d kv_heads=%d hd=%d S=%d batch=%d", heads, kv_heads, hd,
                          S, batch);
    const size_t full = (size_t)heads * hd * S;
    if (!q_stride) q_stride = full;
    if (!k_stride) k_stride = full;
    if (!v_stride) v_stride = full;
    if (q_stride < full || k_stride < full || v_stride < full)
        return mi355_fail("attn_grads_finish: sequence stride below heads*hd*S = %zu", full);
    const int ratio = heads / kv_heads;
    const bool in_place = (const void *)dq == dq_full || (const void *)dk == dk_full || (const void *)dv == dv_full;
    const size_t pairs = (size_t)(heads + 2 * kv_heads) * (hd / 2);        // of one sequence
    auto launch = [&](auto kernel, auto *q, auto *k, auto *v, int vec) {
        const size_t lanes = pairs * ceil_div((size_t)S, (size_t)vec);
        const int per = (int)std::min<size_t>(std::max<size_t>(ST_LANES / lanes, 1), (size_t)batch);   // sequences of one launch
        const size_t kv_full = (size_t)kv_heads * hd * S;
        static_assert(ST_LANES < 1ull << 32, "a launch's lanes are counted in 32 bits");
        for (int b = 0; b < batch; b += std::min(per, batch - b)) {
            const int n = std::min(per, batch - b);
            hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(lanes * n, ST_THREADS)), dim3(ST_THREADS), 0, g_ctx.stream,
                               q + b * q_stride, k + b * k_stride, v + b * v_stride, S, hd, heads, kv_heads, ratio, n,
                               (unsigned)(lanes * n), cos_dev, sin_dev, q_stride, k_stride, v_stride, dq + b * full,
                               dk + b * kv_full, dv + b * kv_full);
        }
    };
    // fp32 without the tables is written as quickly or quicker with streaming stores where three heads and more go into one
    // ([16][2048][256], 16 heads to a KV head, 35 and 27 us, eight heads 29.3 and 26.6; with the tables 25.7 and 25.4, from fp16 21.2 and 21.3)
    const bool far = far_rows(dq, 4 * (size_t)S, 4 * (size_t)S, (size_t)batch * heads * hd) &&
                     (((uintptr_t)dk | (uintptr_t)dv) & 127u) == 0 && (in_f16 || cos_dev || ratio <= 2);
    auto finish = [&](auto vec, auto wave, auto written_through, auto *q, auto *k, auto *v) {
        typedef typename std::remove_const<typename std::remove_pointer<decltype(q)>::type>::type T;
        constexpr int VEC = decltype(vec)::value;
        constexpr bool WAVE = decltype(wave)::value, FAR = decltype(written_through)::value;
        if (cos_dev && ratio == 1) launch(attn_grads_finish_kernel<T, VEC, true, true, WAVE, FAR>, q, k, v, VEC);
        else if (cos_dev) launch(attn_grads_finish_kernel<T, VEC, true, false, WAVE, FAR>, q, k, v, VEC);
        else if (ratio == 1) launch(attn_grads_finish_kernel<T, VEC, false, true, WAVE, FAR>, q, k, v, VEC);
        else launch(attn_grads_finish_kernel<T, VEC, false, false, WAVE, FAR>, q, k, v, VEC);
    };
    auto pick = [&](auto *q, auto *k, auto *v) {
        const std::integral_constant<int, 4> four;
        const std::integral_constant<int, 1> one;
        if (S % 256 == 0 && far) finish(four, std::true_type(), std::true_type(), q, k, v);
        else if (S % 256 == 0) finish(four, std::true_type(), std::false_type(), q, k, v);
        else if (S % 4 == 0 || (S > 4 && !in_place)) finish(four, std::false_type(), std::false_type(), q, k, v);
        else finish(one, std::false_type(), std::false_type(), q, k, v);
    };
    if (in_f16) pick((const _Float16 *)dq_full, (const _Float16 *)dk_full, (const _Float16 *)dv_full);
    else pick((const float *)dq_full, (const float *)dk_full, (const float *)dv_full);
    LAUNCH_OK("attn_grads_finish");
    return 0;
}
