// qknorm_rope.hip — Qwen3 per-head QK-RMSNorm fused with RoPE, forward and backward, one HBM pass.
//
// Not present in the reference: forward = rmsnorm (training/stories_cpu_ops.h:6-21) on each head's
// [hd,S] slab with a [hd] weight shared by the heads, then the forward rotation of interleaved row
// pairs (training/forward.h:55-70, training/training_dynamic/mil_dynamic.h:131-168); backward = the
// inverse rotation (training/training_dynamic/cpu_ops.h:168-184) then rmsnorm_bwd per head
// (training/stories_cpu_ops.h:23-53).
//
// A workgroup owns one head slab x a strip of LPR*4 columns.  Each thread owns whole row PAIRS
// (2i, 2i+1), so the rotation needs no cross-lane traffic; the norm reduction over the hd rows
// uses the same shuffle + LDS exchange as the RMSNorm kernels.
#include "common.h"
#include "tile.h"

namespace {

// ROWS: the tile holds every row pair of the head and nothing else; rows are not whole cache lines.  Then lanes past the end of a row
// load its last columns again, no load is behind a condition, and lines that two pieces share stay in the caches.  us, before / with:
// [22][24 x 128][147] forward 29.5 / 23.7 (cold operands 30.1 / 27.8), backward 41.1 / 32.6 (40.3 / 33.9); [5][570] 25.2 / 19.8 (25.3 /
// 22.7) and 32.7 / 26.3 (32.0 / 28.8); [2][197] 7.7 / 5.4 and 8.5 / 7.3.
template <bool ROWS>
__device__ __forceinline__ v4f qk_load(const float *p) { return ROWS ? ld4(p) : ld4_nt(p); }

template <int LPR, int THREADS, int CAP, bool ROWS = false>
__global__ __launch_bounds__(THREADS) void qknorm_rope_fwd_kernel(
    float *__restrict__ q_out, float *__restrict__ k_out, const float *__restrict__ q, const float *__restrict__ k,
    const float *__restrict__ wq, const float *__restrict__ wk, int hd, int S, int strips, int nq,
    const float *__restrict__ cos_t, const float *__restrict__ sin_t, float eps, float invhd) {
    constexpr int PPS = THREADS / LPR;   // row pairs per step
    constexpr int W = LPR * 4;
    constexpr int NW = THREADS / 64;
    __shared__ float lds[NW * LPR * 4];
    int blk = blockIdx.x;
    const float *in, *w;
    float *out;
    if (blk < nq) { in = q; out = q_out; w = wq; }
    else { blk -= nq; in = k; out = k_out; w = wk; }
    const int slab = blk / strips, strip = blk - slab * strips;
    const int lc = threadIdx.x % LPR, p0 = threadIdx.x / LPR;
    const LaneCols mine = ROWS ? lane_cols_inside<4, W>(strip * W + lc * 4, S) : lane_cols<4>(strip * W + lc * 4, S);
    const int col = mine.col;
    const bool col_ok = mine.ok;
    const int half = hd >> 1;
    const size_t base = (size_t)slab * hd * S + col;

    v4f x0[CAP], x1[CAP];
    float w0[CAP], w1[CAP];
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < CAP; kk++) {
        const int rp = p0 + kk * PPS;
        if (ROWS || (rp < half && col_ok)) {
            const float *px = in + base + (size_t)(2 * rp) * S;
            x0[kk] = qk_load<ROWS>(px);
            x1[kk] = qk_load<ROWS>(px + S);
            w0[kk] = w[2 * rp];
            w1[kk] = w[2 * rp + 1];
        } else {
            x0[kk] = x1[kk] = zero;
            w0[kk] = w1[kk] = 0.f;
        }
    }
    float acc[1][4] = {{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int kk = 0; kk < CAP; kk++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[0][j] += x0[kk][j] * x0[kk][j];
            acc[0][j] += x1[kk][j] * x1[kk][j];
        }
    strip_reduce<4, LPR, THREADS, 1>(acc, lds);
    v4f rr;
#pragma unroll
    for (int j = 0; j < 4; j++) rr[j] = 1.0f / sqrtf(acc[0][j] * invhd + eps);
#pragma unroll
    for (int kk = 0; kk < CAP; kk++) {
        const int rp = p0 + kk * PPS;
        if (ROWS || (rp < half && col_ok)) {
            // the tables are shared by every head and sequence (cache-resident): read here, after the reduction,
            // rather than held in registers across it
            const v4f cs = ld4(cos_t + (size_t)rp * S + col), sn = ld4(sin_t + (size_t)rp * S + col);
            const v4f y0 = (x0[kk] * rr) * w0[kk];
            const v4f y1 = (x1[kk] * rr) * w1[kk];
            float *po = out + base + (size_t)(2 * rp) * S;
            if (!ROWS || col_ok) {
                st4_nt(po, y0 * cs - y1 * sn);
                st4_nt(po + S, y0 * sn + y1 * cs);
            }
        }
    }
}

enum { QK_SOME, QK_ROWS, QK_ALL };
// WHOLE = QK_ALL: the tile holds every row pair of the head and nothing else, every strip is whole: no load or store is behind a condition
// ([16][24 x 128][256] 32.4 -> 31.5 us).  (The forward is slower so, 20.3 -> 21.5: fewer registers, more workgroups at a time.)
template <int LPR, int THREADS, int CAP, int WHOLE = QK_SOME>
__global__ __launch_bounds__(THREADS) void qknorm_rope_bwd_kernel(
    float *dq, float *dk, float *__restrict__ part, const float *dq_out, const float *dk_out,
    const float *__restrict__ q, const float *__restrict__ k, const float *__restrict__ wq,
    const float *__restrict__ wk, int hd, int S, int strips, int nq, const float *__restrict__ cos_t,
    const float *__restrict__ sin_t, float eps, float invhd, int variant) {
    constexpr bool ALL = WHOLE == QK_ALL, ROWS = WHOLE == QK_ROWS;
    constexpr int PPS = THREADS / LPR;
    constexpr int W = LPR * 4;
    constexpr int NW = THREADS / 64;
    __shared__ float lds[NW * 2 * LPR * 4];
    int blk = blockIdx.x;
    float *prt = part + (size_t)blk * hd;
    const float *gin, *xin, *w;
    float *out;
    if (blk < nq) { gin = dq_out; xin = q; out = dq; w = wq; }
    else { blk -= nq; gin = dk_out; xin = k; out = dk; w = wk; }
    const int slab = blk / strips, strip = blk - slab * strips;
    const int lc = threadIdx.x % LPR, p0 = threadIdx.x / LPR;
    const LaneCols mine = ROWS ? lane_cols_inside<4, W>(strip * W + lc * 4, S) : lane_cols<4>(strip * W + lc * 4, S);
    const int col = mine.col;
    const bool col_ok = mine.ok;
    const int half = hd >> 1;
    const size_t base = (size_t)slab * hd * S + col;

    v4f x0[CAP], x1[CAP], d0[CAP], d1[CAP];
    float w0[CAP], w1[CAP];
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < CAP; kk++) {
        const int rp = p0 + kk * PPS;
        if (ALL || ROWS || (rp < half && col_ok)) {
            const size_t o = base + (size_t)(2 * rp) * S;
            x0[kk] = qk_load<ROWS>(xin + o);
            x1[kk] = qk_load<ROWS>(xin + o + S);
            const v4f g0 = qk_load<ROWS>(gin + o), g1 = qk_load<ROWS>(gin + o + S);
            const v4f c = ld4(cos_t + (size_t)rp * S + col), s = ld4(sin_t + (size_t)rp * S + col);
            d0[kk] = g0 * c + g1 * s;        // inverse rotation (cpu_ops.h:179-180)
            d1[kk] = (-g0) * s + g1 * c;
            w0[kk] = w[2 * rp];
            w1[kk] = w[2 * rp + 1];
        } else {
            x0[kk] = x1[kk] = d0[kk] = d1[kk] = zero;
            w0[kk] = w1[kk] = 0.f;
        }
    }
    float acc[2][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int kk = 0; kk < CAP; kk++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[0][j] += x0[kk][j] * x0[kk][j];
            acc[0][j] += x1[kk][j] * x1[kk][j];
            acc[1][j] += (d0[kk][j] * x0[kk][j]) * w0[kk];
            acc[1][j] += (d1[kk][j] * x1[kk][j]) * w1[kk];
        }
    strip_reduce<4, LPR, THREADS, 2>(acc, lds);
    v4f rr, dotn;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        rr[j] = 1.0f / sqrtf(acc[0][j] * invhd + eps);
        dotn[j] = acc[1][j] * ((rr[j] * rr[j]) * invhd);
    }
#pragma unroll
    for (int kk = 0; kk < CAP; kk++) {
        const int rp = p0 + kk * PPS;
        if (ALL || ROWS || rp < half) {   // uniform over each group of LPR lanes
            v4f o0, o1;
            if (variant == 0) {
                o0 = ((d0[kk] - x0[kk] * dotn) * rr) * w0[kk];
                o1 = ((d1[kk] - x1[kk] * dotn) * rr) * w1[kk];
            } else {
                o0 = (d0[kk] * w0[kk]) * rr - (x0[kk] * dotn) * rr;
                o1 = (d1[kk] * w1[kk]) * rr - (x1[kk] * dotn) * rr;
            }
            if (ALL || col_ok) {
                float *po = out + base + (size_t)(2 * rp) * S;
                st4_nt(po, o0);
                st4_nt(po + S, o1);
            }
            const v4f t0 = (d0[kk] * x0[kk]) * rr, t1 = (d1[kk] * x1[kk]) * rr;
            float s0 = own_sum<4>(mine, [&](int j) { return t0[j]; });
            float s1 = own_sum<4>(mine, [&](int j) { return t1[j]; });
            s0 = group_sum<LPR>(s0);
            s1 = group_sum<LPR>(s1);
            if (lc == 0) {
                prt[2 * rp] = s0;
                prt[2 * rp + 1] = s1;
            }
        }
    }
}

// measured at the Qwen3 shape: 8-wave workgroups (two pairs per lane, 5 waves per SIMD) run the backward
// 7 % faster than 4-wave ones (four pairs per lane, 2 waves per SIMD); the forward does not care
constexpr int QK_THREADS_FWD = 256, QK_THREADS_BWD = 512;

struct QkCfg {
    int lpr, threads, cap;
};

// Widest strip whose row pairs fit the register tile (at most 4 pairs per lane: 8 would spill).  In place the short
// last group of columns of a row and its neighbour must lie in one strip (lane_cols in tile.h).
bool pick_qk(int hd, int S, bool in_place, QkCfg &cfg, bool backward) {
    const int half = hd / 2;
    if (S < 4) return false;
    const int lprs[3] = {16, 8, 4};
    const int thr = g_ctx.qk_threads == 256 || g_ctx.qk_threads == 512 ? g_ctx.qk_threads : (backward ? QK_THREADS_BWD : QK_THREADS_FWD);
    for (int lpr : lprs) {
        if (g_ctx.qk_lpr && g_ctx.qk_lpr != lpr) continue;
        if (in_place && !tail_in_strip(S, lpr * 4, 4)) continue;
        const int pps = thr / lpr;
        const int caps[3] = {1, 2, 4};
        for (int cap : caps)
            if (cap * pps >= half) { cfg = QkCfg{lpr, thr, cap}; return true; }
    }
    return false;
}

#define QK_DISPATCH(KERNEL, cfg, grid, ...)                                                                   \
    do {                                                                                                      \
        const int key = (cfg).lpr * 10000 + ((cfg).threads / 256) * 100 + (cfg).cap;                          \
        switch (key) {                                                                                        \
            case 160101: hipLaunchKernelGGL((KERNEL<16, 256, 1>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 160102: hipLaunchKernelGGL((KERNEL<16, 256, 2>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 160104: hipLaunchKernelGGL((KERNEL<16, 256, 4>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 160201: hipLaunchKernelGGL((KERNEL<16, 512, 1>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 160202: hipLaunchKernelGGL((KERNEL<16, 512, 2>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 160204: hipLaunchKernelGGL((KERNEL<16, 512, 4>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 80101: hipLaunchKernelGGL((KERNEL<8, 256, 1>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 80102: hipLaunchKernelGGL((KERNEL<8, 256, 2>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 80104: hipLaunchKernelGGL((KERNEL<8, 256, 4>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 80201: hipLaunchKernelGGL((KERNEL<8, 512, 1>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 80202: hipLaunchKernelGGL((KERNEL<8, 512, 2>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 80204: hipLaunchKernelGGL((KERNEL<8, 512, 4>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 40101: hipLaunchKernelGGL((KERNEL<4, 256, 1>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 40102: hipLaunchKernelGGL((KERNEL<4, 256, 2>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 40104: hipLaunchKernelGGL((KERNEL<4, 256, 4>), grid, dim3(256), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 40201: hipLaunchKernelGGL((KERNEL<4, 512, 1>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 40202: hipLaunchKernelGGL((KERNEL<4, 512, 2>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            case 40204: hipLaunchKernelGGL((KERNEL<4, 512, 4>), grid, dim3(512), 0, g_ctx.stream, __VA_ARGS__); break; \
            default: return mi355_fail("qknorm_rope: no kernel for tile key %d", key);                        \
        }                                                                                                     \
    } while (0)

// Rows that are not whole 128-byte lines, on a tile that the head's row pairs fill (hd 128 and 64): the ROWS kernels.
bool whole_rows(const QkCfg &cfg, int hd, int S) { return S % 32 != 0 && cfg.lpr == 16 && cfg.threads / 16 * cfg.cap * 2 == hd; }
// Where the forward is quicker with them, by the workgroups to a compute unit.  The other kernel does best just before its workgroups
// need another round: hd 64 from four to five of them ([12][24 x 64][197] 10.5 us, ROWS 12.3; six, [16], 15.3 and 13.9), hd 128 from
// three to four ([12][24 x 128][147] 16.0, 17.1; three, [16][24 x 128][100], 13.5, 13.0).  Lanes past the end of a row ask for what others
// have: in a single strip that costs more than it saves from three on ([64][24 x 64][54] 9.7, 11.3; [32][24 x 128][54] 9.2, 10.7;
// [4][24 x 128][54] 6.2, 4.4), and in two of which the second is nearly empty from six on ([30][24 x 64][70] 1.15 times as long).
bool forward_rows(int hd, int S, size_t workgroups) {
    const size_t cus = g_ctx.num_cu > 0 ? g_ctx.num_cu : 256, round = ceil_div(workgroups, cus);
    return round != (hd == 128 ? 4 : 5) && (S >= 80 || round <= (S <= 64 ? 2 : 5));
}

int check_shape(const char *who, int heads, int kv_heads, int hd, int S, int batch) {
    if (hd <= 0 || (hd & 1) || S <= 0 || batch <= 0 || heads < 0 || kv_heads < 0 || heads + kv_heads == 0)
        return mi355_fail("%s: bad shape heads=%d kv_heads=%d hd=%d S=%d batch=%d", who, heads, kv_heads, hd, S, batch);
    return 0;
}

}   // namespace

MI355_API int mi355_qknorm_rope_fwd_dev(float *q_out, float *k_out, const float *q, const float *k, const float *wq,
                                        const float *wk, int heads, int kv_heads, int hd, int S, int batch,
                                        const float *cos_dev, const float *sin_dev, float eps) {
    if (!mi355_ready("qknorm_rope_fwd")) return -1;
    if (check_shape("qknorm_rope_fwd", heads, kv_heads, hd, S, batch)) return -1;
    if (!cos_dev || !sin_dev || (heads > 0 && (!q_out || !q || !wq)) || (kv_heads > 0 && (!k_out || !k || !wk)))
        return mi355_fail("qknorm_rope_fwd: NULL pointer");
    QkCfg cfg;
    if (!pick_qk(hd, S, (heads > 0 && q_out == q) || (kv_heads > 0 && k_out == k), cfg, false)) {
        // unfused composition: per-head norm (heads folded into the batch), then the rotation in place
        if (heads > 0 && mi355_rmsnorm_fwd_dev(q_out, q, wq, hd, S, batch * heads, eps)) return -1;
        if (kv_heads > 0 && mi355_rmsnorm_fwd_dev(k_out, k, wk, hd, S, batch * kv_heads, eps)) return -1;
        return mi355_rope_dev(q_out, k_out, q_out, k_out, heads, kv_heads, hd, S, batch, cos_dev, sin_dev, +1);
    }
    const int strips = (int)ceil_div((size_t)S, (size_t)cfg.lpr * 4);
    const int nq = batch * heads * strips, nk = batch * kv_heads * strips;
    auto launch = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, dim3(nq + nk), dim3(threads), 0, g_ctx.stream, q_out, k_out, q, k, wq, wk, hd, S, strips, nq, cos_dev,
                           sin_dev, eps, 1.0f / (float)hd);
    };
    const bool rows = whole_rows(cfg, hd, S) && forward_rows(hd, S, (size_t)(nq + nk));
    if (rows && cfg.threads == 256 && cfg.cap == 4) launch(qknorm_rope_fwd_kernel<16, 256, 4, true>, 256);
    else if (rows && cfg.threads == 256 && cfg.cap == 2) launch(qknorm_rope_fwd_kernel<16, 256, 2, true>, 256);
    else
        QK_DISPATCH(qknorm_rope_fwd_kernel, cfg, dim3(nq + nk), q_out, k_out, q, k, wq, wk, hd, S, strips, nq, cos_dev,
                    sin_dev, eps, 1.0f / (float)hd);
    LAUNCH_OK("qknorm_rope_fwd");
    return 0;
}

MI355_API int mi355_qknorm_rope_bwd_dev(float *dq, float *dk, float *dwq, float *dwk, const float *dq_out,
                                        const float *dk_out, const float *q, const float *k, const float *wq,
                                        const float *wk, int heads, int kv_heads, int hd, int S, int batch,
                                        const float *cos_dev, const float *sin_dev, float eps, int variant) {
    if (!mi355_ready("qknorm_rope_bwd")) return -1;
    if (check_shape("qknorm_rope_bwd", heads, kv_heads, hd, S, batch)) return -1;
    if (variant != 0 && variant != 1) return mi355_fail("qknorm_rope_bwd: variant must be 0 or 1");
    if (!cos_dev || !sin_dev || (heads > 0 && (!dq || !dwq || !dq_out || !q || !wq)) ||
        (kv_heads > 0 && (!dk || !dwk || !dk_out || !k || !wk)))
        return mi355_fail("qknorm_rope_bwd: NULL pointer");
    QkCfg cfg;
    if (!pick_qk(hd, S, (heads > 0 && dq == dq_out) || (kv_heads > 0 && dk == dk_out), cfg, true)) {
        // unfused composition: inverse rotation into dq/dk, then the per-head norm backward in place
        if (mi355_rope_dev(dq, dk, dq_out, dk_out, heads, kv_heads, hd, S, batch, cos_dev, sin_dev, -1)) return -1;
        if (heads > 0 && mi355_rmsnorm_bwd_dev(dq, dwq, dq, q, wq, hd, S, batch * heads, eps, variant)) return -1;
        if (kv_heads > 0 && mi355_rmsnorm_bwd_dev(dk, dwk, dk, k, wk, hd, S, batch * kv_heads, eps, variant)) return -1;
        return 0;
    }
    const int strips = (int)ceil_div((size_t)S, (size_t)cfg.lpr * 4);
    const int nq = batch * heads * strips, nk = batch * kv_heads * strips;
    float *part = mi355_dw_partials((size_t)(nq + nk) * hd, nq > 0 ? dwq : nullptr, nk > 0 ? dwk : nullptr);
    if (!part) return -1;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nq + nk), dim3(512), 0, g_ctx.stream, dq, dk, part, dq_out, dk_out, q, k, wq, wk, hd, S, strips, nq,
                           cos_dev, sin_dev, eps, 1.0f / (float)hd, variant);
    };
    const bool rows = whole_rows(cfg, hd, S);
    if (cfg.lpr == 16 && cfg.threads == 512 && cfg.cap == 2 && hd == 128 && S % 64 == 0)
        launch(qknorm_rope_bwd_kernel<16, 512, 2, QK_ALL>);
    else if (rows && cfg.threads == 512 && cfg.cap == 2) launch(qknorm_rope_bwd_kernel<16, 512, 2, QK_ROWS>);
    else if (rows && cfg.threads == 512 && cfg.cap == 1) launch(qknorm_rope_bwd_kernel<16, 512, 1, QK_ROWS>);
    else
        QK_DISPATCH(qknorm_rope_bwd_kernel, cfg, dim3(nq + nk), dq, dk, part, dq_out, dk_out, q, k, wq, wk, hd, S, strips,
                    nq, cos_dev, sin_dev, eps, 1.0f / (float)hd, variant);
    LAUNCH_OK("qknorm_rope_bwd");
    if (nq > 0 && mi355_dw_submit(dwq, part, nq, hd)) return -1;
    if (nk > 0 && mi355_dw_submit(dwk, part + (size_t)nq * hd, nk, hd)) return -1;
    return mi355_dw_op_end();
}
