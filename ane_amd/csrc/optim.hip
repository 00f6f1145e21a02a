// optim.hip — the optimizer tail of the training loops: gradient scale, global L2 norm, clip, Adam/AdamW.
//
// Reference: training/training_dynamic/train.m:748-877 — a scale pass over every gradient (:754-769),
// vDSP_dotpr per tensor for the global norm (:771-787), a clip pass (:806-821), adam_update per tensor
// (training/training_dynamic/cpu_ops.h:56-64; wd = 0 is training/stories_cpu_ops.h:55-63) and a zeroing
// pass (:873-877).  That is five sweeps over the gradients; here it is two: one read for the norm
// (with the scale folded in) and one fused update that applies both scales, updates m, v, w and can
// clear the gradient in the same pass.  Pure HBM streams: 16 B read + 12-16 B written per parameter.
#include "common.h"

#include <math.h>
#include <algorithm>

namespace {

constexpr int OPT_THREADS = 256;

// fixed grid -> fixed assignment of elements to lanes -> deterministic sum
__global__ __launch_bounds__(OPT_THREADS) void sumsq_partial_kernel(float *__restrict__ part,
                                                                    const float *__restrict__ g, size_t n, size_t n4,
                                                                    float pre, bool vec) {
    __shared__ float red[OPT_THREADS / 64];
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    const size_t tid = (size_t)blockIdx.x * OPT_THREADS + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * OPT_THREADS;
    if (vec) {
        for (size_t i = tid; i < n4; i += stride) {
            v4f v = ld4_nt(g + 4 * i) * pre;            // the scale pass of train.m:755-769, folded in
            s0 += v.x * v.x; s1 += v.y * v.y; s2 += v.z * v.z; s3 += v.w * v.w;
        }
        if (blockIdx.x == 0)
            for (size_t i = n4 * 4 + threadIdx.x; i < n; i += OPT_THREADS) { float t = g[i] * pre; s0 += t * t; }
    } else {
        for (size_t i = tid; i < n; i += stride) { float t = g[i] * pre; s0 += t * t; }
    }
    float s = (s0 + s1) + (s2 + s3);
    s = wave_sum_far_first(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(1024) void sumsq_final_kernel(float *__restrict__ acc, const float *__restrict__ part,
                                                           int nblk) {
    __shared__ float red[1024];
    float s = 0.f;
    for (int i = threadIdx.x; i < nblk; i += 1024) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) *acc = *acc + red[0];
}

// clip_scale = grad_clip / sqrt(sumsq) when clipping applies, else 1 (train.m:806-808)
__global__ void clip_scale_kernel(float *scale, const float *sumsq, float grad_clip) {
    const float norm = sqrtf(*sumsq);
    *scale = (grad_clip > 0.f && norm > grad_clip) ? grad_clip / norm : 1.0f;
}

__device__ __forceinline__ void adam1(float &w, float &m, float &v, float g, float lr, float b1, float b2,
                                      float omb1, float omb2, float eps, float wd, float bc1, float bc2) {
    // cpu_ops.h:59-62, one rounding per operation
    m = b1 * m + omb1 * g;
    v = b2 * v + (omb2 * g) * g;
    const float mh = m / bc1, vh = v / bc2;
    w -= lr * (mh / (sqrtf(vh) + eps) + wd * w);
}

template <bool ZERO, int THREADS>
__global__ __launch_bounds__(THREADS) void adam_kernel(float *__restrict__ w, float *__restrict__ g,
                                                           float *__restrict__ m, float *__restrict__ v, size_t n,
                                                           size_t n4, float lr, float b1, float b2, float eps,
                                                           float wd, float bc1, float bc2, float scale1,
                                                           const float *__restrict__ scale2_p, bool vec) {
    const float scale2 = scale2_p ? *scale2_p : 1.0f;
    const float omb1 = 1.0f - b1, omb2 = 1.0f - b2;
    const size_t i = (size_t)blockIdx.x * THREADS + threadIdx.x;
    if (vec) {
        if (i < n4) {
            v4f wv = ld4_nt(w + 4 * i), gv = ld4_nt(g + 4 * i), mv = ld4_nt(m + 4 * i), vv = ld4_nt(v + 4 * i);
            gv = (gv * scale1) * scale2;                 // the two scale passes (train.m:755-769, 806-821)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float a = wv[j], b = mv[j], c = vv[j];
                adam1(a, b, c, gv[j], lr, b1, b2, omb1, omb2, eps, wd, bc1, bc2);
                wv[j] = a; mv[j] = b; vv[j] = c;
            }
            st4_stream(w + 4 * i, wv, THREADS == FAR_THREADS);
            st4_stream(m + 4 * i, mv, THREADS == FAR_THREADS);
            st4_stream(v + 4 * i, vv, THREADS == FAR_THREADS);
            if (ZERO) { const v4f z = {0.f, 0.f, 0.f, 0.f}; st4_stream(g + 4 * i, z, THREADS == FAR_THREADS); }
        }
        if (blockIdx.x == 0 && threadIdx.x < n - n4 * 4) {
            const size_t k = n4 * 4 + threadIdx.x;
            float gg = (g[k] * scale1) * scale2;
            adam1(w[k], m[k], v[k], gg, lr, b1, b2, omb1, omb2, eps, wd, bc1, bc2);
            if (ZERO) g[k] = 0.f;
        }
    } else if (i < n) {
        float gg = (g[i] * scale1) * scale2;
        adam1(w[i], m[i], v[i], gg, lr, b1, b2, omb1, omb2, eps, wd, bc1, bc2);
        if (ZERO) g[i] = 0.f;
    }
}

// The same update from arrays to others: from the pinned block of a call on host arrays to that of its results, over the link (stream()
// in host_stage.h has the times).
__global__ __launch_bounds__(OPT_THREADS) void adam_between_kernel(float *__restrict__ wo, float *__restrict__ mo, float *__restrict__ vo,
                                                                   const float *__restrict__ w, const float *__restrict__ g,
                                                                   const float *__restrict__ m, const float *__restrict__ v, size_t n,
                                                                   size_t n4, float lr, float b1, float b2, float eps, float wd,
                                                                   float bc1, float bc2) {
    const float omb1 = 1.0f - b1, omb2 = 1.0f - b2;
    const size_t i = (size_t)blockIdx.x * OPT_THREADS + threadIdx.x;
    if (i < n4) {
        v4f wv = ld4_nt(w + 4 * i), gv = ld4_nt(g + 4 * i), mv = ld4_nt(m + 4 * i), vv = ld4_nt(v + 4 * i);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float a = wv[j], b = mv[j], c = vv[j];
            adam1(a, b, c, gv[j], lr, b1, b2, omb1, omb2, eps, wd, bc1, bc2);
            wv[j] = a; mv[j] = b; vv[j] = c;
        }
        st4_nt(wo + 4 * i, wv);
        st4_nt(mo + 4 * i, mv);
        st4_nt(vo + 4 * i, vv);
    }
    if (blockIdx.x == 0 && threadIdx.x < n - n4 * 4) {
        const size_t k = n4 * 4 + threadIdx.x;
        float a = w[k], b = m[k], c = v[k];
        adam1(a, b, c, g[k], lr, b1, b2, omb1, omb2, eps, wd, bc1, bc2);
        wo[k] = a; mo[k] = b; vo[k] = c;
    }
}

// ---- many tensors per launch ----
// The blocks of all tensors of a launch are numbered through: tensor i owns the blocks first[i] .. first[i + 1] - 1.
// A grid of (blocks of the largest tensor) x (tensors) is mostly empty workgroups where sizes differ: the 110 M
// parameters of 12 layers and an embedding started 460 000 workgroups for 108 000 that had work.
constexpr int MT_MAX = 64;                  // 3.1 KB of kernel arguments (4 KB is the most a launch takes)
constexpr int SQ_V4 = 8;                    // 128-bit loads of a lane of the norm, all in flight together
struct MtFirst {
    unsigned first[MT_MAX];                 // 2^32 - 1 behind the last tensor
};
struct MtSumsq {
    MtFirst blk;
    const float *g[MT_MAX];
    size_t n[MT_MAX];
};
struct MtAdam {
    MtFirst blk;
    float *w[MT_MAX], *g[MT_MAX], *m[MT_MAX], *v[MT_MAX];
    size_t n[MT_MAX];
    float wd[MT_MAX];
};

// The tensor that owns a block: two rounds of eight comparisons on scalar registers, two trips to the scalar cache
// (a search by halves would be six dependent trips ahead of the first load of data).
__device__ __forceinline__ int mt_owner(const MtFirst &f, unsigned block) {
    int g = 0;
#pragma unroll
    for (int j = 1; j < MT_MAX / 8; j++) g += block >= f.first[8 * j] ? 1 : 0;
    int i = 0;
#pragma unroll
    for (int j = 1; j < 8; j++) i += block >= f.first[8 * g + j] ? 1 : 0;
    return 8 * g + i;
}

// One partial per block, in block order.  Bound by the read of g (110 M floats: 438 MB).  The loads are ordinary ones,
// so that the end of g is in the 256 MB last-level cache when the update, which walks the blocks from the last to the
// first, asks for it.  Norm + clip + update of the 110 M parameters (109 tensors, 3.5 GB besides the norm's read):
// 748 us with one launch per 16 tensors of (largest tensor) x (tensors) blocks and a sum after each, 707 with the
// blocks numbered through, 700 with the update backwards, 650 with these loads not marked as streaming.  Which elements
// a block sums depends on the sizes alone, so the sum is deterministic.
__global__ __launch_bounds__(OPT_THREADS) void sumsq_partial_mt_kernel(float *__restrict__ part, MtSumsq a, float pre,
                                                                       int rounds) {
    __shared__ float red[OPT_THREADS / 64];
    const int ti = mt_owner(a.blk, blockIdx.x);
    const float *__restrict__ g = a.g[ti];
    const size_t n = a.n[ti], n4 = n / 4;
    size_t i0 = (size_t)(blockIdx.x - a.blk.first[ti]) * rounds * (OPT_THREADS * SQ_V4) + threadIdx.x;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    for (int r = 0; r < rounds; r++, i0 += OPT_THREADS * SQ_V4) {
        v4f v[SQ_V4];
#pragma unroll
        for (int k = 0; k < SQ_V4; k++) {
            const size_t i = i0 + (size_t)k * OPT_THREADS;
            v[k] = i < n4 ? ld4(g + 4 * i) : v4f{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int k = 0; k < SQ_V4; k++) {
            const v4f t = v[k] * pre;
            s0 += t.x * t.x; s1 += t.y * t.y; s2 += t.z * t.z; s3 += t.w * t.w;
        }
#pragma unroll
        for (int k = 0; k < SQ_V4; k++)
            if (i0 + (size_t)k * OPT_THREADS == n4)              // the lane behind the last whole group
                for (size_t j = 4 * n4; j < n; j++) { const float t = g[j] * pre; s0 += t * t; }
    }
    float s = (s0 + s1) + (s2 + s3);
    s = wave_sum_far_first(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Bound by its eight streams (16 B read, 16 B written per parameter with ZERO, at the 5.7 TB/s of a copy).  Norm + clip + update of
// the 110 M parameters: 650 us in workgroups of 256 with streaming stores (of 1024 705, plain stores 725, g read and cleared with
// ordinary accesses 698), 630 a wave to a workgroup with stores written through.
// THREADS == FAR_THREADS: that form, for launches of MT_FAR parameters and more whose tensors all start on a line.  The update alone, us,
// in workgroups of 256 / so: 110 M with the embedding 605 / 576, layers of 7.1 M parameters without it, seven 280 / 270, three 117 / 115,
// one 40.5 / 40.7 (with g kept instead of cleared 35 / 35, 97 / 98, seven 227 / 229), 64 tensors of 64 K 25.4 / 26.5.  Starts
// 16 bytes into a line, whose lines a wave writes in two pieces: 110 M 703 / 766, two tensors of 8 M 103 / 118, 64 of 64 K 27.7 / 32.
constexpr size_t MT_FAR = (size_t)16 << 20;
template <bool ZERO, int THREADS>
__global__ __launch_bounds__(THREADS) void adam_mt_kernel(MtAdam a, float lr, float b1, float b2, float eps,
                                                              float bc1, float bc2, float scale1,
                                                              const float *__restrict__ scale2_p) {
    const unsigned block = gridDim.x - 1 - blockIdx.x;
    const int ti = mt_owner(a.blk, block);
    const size_t n = a.n[ti], n4 = n / 4;
    const size_t i = (size_t)(block - a.blk.first[ti]) * THREADS + threadIdx.x;
    float *__restrict__ w = a.w[ti], *__restrict__ g = a.g[ti];
    float *__restrict__ m = a.m[ti], *__restrict__ v = a.v[ti];
    const float wd = a.wd[ti];
    const float scale2 = scale2_p ? *scale2_p : 1.0f;
    const float omb1 = 1.0f - b1, omb2 = 1.0f - b2;
    if (i < n4) {
        v4f wv = ld4_nt(w + 4 * i), gv = ld4_nt(g + 4 * i), mv = ld4_nt(m + 4 * i), vv = ld4_nt(v + 4 * i);
        gv = (gv * scale1) * scale2;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float x = wv[j], y = mv[j], z = vv[j];
            adam1(x, y, z, gv[j], lr, b1, b2, omb1, omb2, eps, wd, bc1, bc2);
            wv[j] = x; mv[j] = y; vv[j] = z;
        }
        st4_stream(w + 4 * i, wv, THREADS == FAR_THREADS);
        st4_stream(m + 4 * i, mv, THREADS == FAR_THREADS);
        st4_stream(v + 4 * i, vv, THREADS == FAR_THREADS);
        if (ZERO) { const v4f z4 = {0.f, 0.f, 0.f, 0.f}; st4_stream(g + 4 * i, z4, THREADS == FAR_THREADS); }
    } else if (i == n4) {
        for (size_t k = 4 * n4; k < n; k++) {                    // fewer than four are left
            const float gg = (g[k] * scale1) * scale2;
            adam1(w[k], m[k], v[k], gg, lr, b1, b2, omb1, omb2, eps, wd, bc1, bc2);
            if (ZERO) g[k] = 0.f;
        }
    }
}

// The block table of the first tensors of a list, `per` 128-bit groups to a block of `threads` (one more group where a tensor
// ends within one): as many as one launch holds (MT_MAX, and fewer than 2^32 threads).  Returns how many; `blocks`: theirs.
int mt_blocks(MtFirst &f, unsigned &blocks, const size_t *n, int count, size_t per, int threads) {
    size_t total = 0;
    int k = 0;
    for (; k < count && k < MT_MAX; k++) {
        const size_t more = ceil_div(ceil_div(n[k], (size_t)4), per);
        if (total + more >= ((size_t)1 << 32) / threads) break;
        f.first[k] = (unsigned)total;
        total += more;
    }
    for (int i = k; i < MT_MAX; i++) f.first[i] = 0xffffffffu;
    blocks = (unsigned)total;
    return k;
}

}   // namespace

MI355_API int mi355_sumsq_accum_multi_dev(float *acc_dev, const float *const *g, const size_t *n, int count,
                                          float pre_scale) {
    if (!mi355_ready("sumsq_accum_multi")) return -1;
    if (!acc_dev || !g || !n || count <= 0) return mi355_fail("sumsq_accum_multi: bad arguments");
    for (int i = 0; i < count; i++)
        if (!g[i] || n[i] == 0 || !aligned16(g[i])) return mi355_fail("sumsq_accum_multi: tensor %d is NULL, empty or not 16-byte aligned", i);
    // from 134 M elements on a block takes several rounds, so that the partials stay near 64 KB
    size_t all = 0, total = 0, done = 0;
    for (int i = 0; i < count; i++) all += n[i] / 4;
    const int rounds = (int)std::min<size_t>(ceil_div(all + 1, (size_t)OPT_THREADS * SQ_V4 * 16384), 1u << 30);
    const size_t per = (size_t)OPT_THREADS * SQ_V4 * rounds;
    for (int i = 0; i < count; i++) total += ceil_div(ceil_div(n[i], (size_t)4), per);
    float *part = (float *)mi355_ws(total * sizeof(float));
    if (!part) return -1;
    for (int i0 = 0, k = 0; i0 < count; i0 += k) {
        MtSumsq a = {};
        unsigned blocks;
        k = mt_blocks(a.blk, blocks, n + i0, count - i0, per, OPT_THREADS);
        if (!k) return mi355_fail("sumsq_accum_multi: tensor %d is too large for one launch", i0);
        for (int i = 0; i < k; i++) { a.g[i] = g[i0 + i]; a.n[i] = n[i0 + i]; }
        hipLaunchKernelGGL(sumsq_partial_mt_kernel, dim3(blocks), dim3(OPT_THREADS), 0, g_ctx.stream, part + done, a, pre_scale,
                           rounds);
        done += blocks;
    }
    hipLaunchKernelGGL(sumsq_final_kernel, dim3(1), dim3(1024), 0, g_ctx.stream, acc_dev, part, (int)total);
    LAUNCH_OK("sumsq_accum_multi");
    return 0;
}

MI355_API int mi355_adam_update_multi_dev(float *const *w, float *const *g, float *const *m, float *const *v,
                                          const size_t *n, const float *wd, int count, int t, float lr, float b1,
                                          float b2, float eps, float scale1, const float *scale2_dev, int zero_grad) {
    if (!mi355_ready("adam_update_multi")) return -1;
    if (!w || !g || !m || !v || !n || !wd || count <= 0 || t < 1) return mi355_fail("adam_update_multi: bad arguments");
    for (int i = 0; i < count; i++)
        if (!w[i] || !g[i] || !m[i] || !v[i] || n[i] == 0 || !aligned16(w[i]) || !aligned16(g[i]) || !aligned16(m[i]) ||
            !aligned16(v[i]))
            return mi355_fail("adam_update_multi: tensor %d is NULL, empty or not 16-byte aligned", i);
    const float bc1 = 1.0f - powf(b1, (float)t), bc2 = 1.0f - powf(b2, (float)t);
    for (int i0 = 0, k = 0; i0 < count; i0 += k) {
        MtAdam a = {};
        unsigned blocks;
        k = mt_blocks(a.blk, blocks, n + i0, count - i0, OPT_THREADS, OPT_THREADS);
        size_t all = 0;
        uintptr_t starts = 0;
        for (int i = i0; i < i0 + k; i++) {
            all += n[i];
            starts |= (uintptr_t)w[i] | (uintptr_t)g[i] | (uintptr_t)m[i] | (uintptr_t)v[i];
        }
        const bool far = all >= MT_FAR && (starts & 127u) == 0;
        if (far) k = mt_blocks(a.blk, blocks, n + i0, count - i0, FAR_THREADS, FAR_THREADS);
        if (!k) return mi355_fail("adam_update_multi: tensor %d is too large for one launch", i0);
        for (int i = 0; i < k; i++) {
            a.w[i] = w[i0 + i]; a.g[i] = g[i0 + i]; a.m[i] = m[i0 + i]; a.v[i] = v[i0 + i];
            a.n[i] = n[i0 + i]; a.wd[i] = wd[i0 + i];
        }
#define ADAM_MT(ZERO, T)                                                                                             \
    hipLaunchKernelGGL((adam_mt_kernel<ZERO, T>), dim3(blocks), dim3(T), 0, g_ctx.stream, a, lr, b1, b2, eps, bc1, bc2, scale1, \
                       scale2_dev)
        if (far) { if (zero_grad) ADAM_MT(true, FAR_THREADS); else ADAM_MT(false, FAR_THREADS); }
        else { if (zero_grad) ADAM_MT(true, OPT_THREADS); else ADAM_MT(false, OPT_THREADS); }
#undef ADAM_MT
        LAUNCH_OK("adam_update_multi");
    }
    return 0;
}

MI355_API int mi355_sumsq_accum_dev(float *acc_dev, const float *g, size_t n, float pre_scale) {
    if (!mi355_ready("sumsq_accum")) return -1;
    if (!acc_dev || !g) return mi355_fail("sumsq_accum: NULL pointer");
    if (n == 0) return mi355_fail("sumsq_accum: empty tensor");
    const bool vec = aligned16(g);
    const size_t n4 = vec ? n / 4 : 0;
    size_t blocks = ceil_div(vec ? (n4 ? n4 : 1) : n, (size_t)OPT_THREADS * 4);
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    float *part = (float *)mi355_ws(blocks * sizeof(float));
    if (!part) return -1;
    hipLaunchKernelGGL(sumsq_partial_kernel, dim3((unsigned)blocks), dim3(OPT_THREADS), 0, g_ctx.stream, part, g, n, n4,
                       pre_scale, vec);
    hipLaunchKernelGGL(sumsq_final_kernel, dim3(1), dim3(1024), 0, g_ctx.stream, acc_dev, part, (int)blocks);
    LAUNCH_OK("sumsq_accum");
    return 0;
}

MI355_API int mi355_clip_scale_dev(float *scale_dev, const float *sumsq_dev, float grad_clip) {
    if (!mi355_ready("clip_scale")) return -1;
    if (!scale_dev || !sumsq_dev) return mi355_fail("clip_scale: NULL pointer");
    hipLaunchKernelGGL(clip_scale_kernel, dim3(1), dim3(1), 0, g_ctx.stream, scale_dev, sumsq_dev, grad_clip);
    LAUNCH_OK("clip_scale");
    return 0;
}

MI355_API int mi355_adam_update_dev(float *w, float *g, float *m, float *v, size_t n, int t, float lr, float b1,
                                    float b2, float eps, float wd, float scale1, const float *scale2_dev,
                                    int zero_grad) {
    if (!mi355_ready("adam_update")) return -1;
    if (!w || !g || !m || !v) return mi355_fail("adam_update: NULL pointer");
    if (n == 0 || t < 1) return mi355_fail("adam_update: empty tensor or step < 1");
    // bias corrections as the reference computes them (cpu_ops.h:57)
    const float bc1 = 1.0f - powf(b1, (float)t), bc2 = 1.0f - powf(b2, (float)t);
    const bool vec = aligned16(w) && aligned16(g) && aligned16(m) && aligned16(v);
    const size_t n4 = vec ? n / 4 : 0;
    const size_t work = vec ? (n4 ? n4 : 1) : n;
    const bool far = 16 * n4 >= FAR_BYTES && (((uintptr_t)w | (uintptr_t)g | (uintptr_t)m | (uintptr_t)v) & 127u) == 0;
#define ADAM(ZERO, T)                                                                                                \
    hipLaunchKernelGGL((adam_kernel<ZERO, T>), dim3((unsigned)ceil_div(work, (size_t)T)), dim3(T), 0, g_ctx.stream, w, g, m, v, n, \
                       n4, lr, b1, b2, eps, wd, bc1, bc2, scale1, scale2_dev, vec)
    if (far) { if (zero_grad) ADAM(true, FAR_THREADS); else ADAM(false, FAR_THREADS); }
    else { if (zero_grad) ADAM(true, OPT_THREADS); else ADAM(false, OPT_THREADS); }
#undef ADAM
    LAUNCH_OK("adam_update");
    return 0;
}

int mi355_adam_between(float *wo, float *mo, float *vo, const float *w, const float *g, const float *m, const float *v, size_t n, int t,
                       float lr, float b1, float b2, float eps, float wd) {
    const float bc1 = 1.0f - powf(b1, (float)t), bc2 = 1.0f - powf(b2, (float)t);
    const size_t n4 = n / 4, blocks = std::max<size_t>(ceil_div(n4, (size_t)OPT_THREADS), 1);
    hipLaunchKernelGGL(adam_between_kernel, dim3((unsigned)blocks), dim3(OPT_THREADS), 0, g_ctx.stream, wo, mo, vo, w, g, m, v, n, n4, lr,
                       b1, b2, eps, wd, bc1, bc2);
    LAUNCH_OK("adam_update");
    return 0;
}
