// gemm.hip — the loops' cblas_sgemm(CblasRowMajor, ...) calls on device memory.
//
// The dynamic loop runs the classifier and every weight-gradient product on the CPU through cblas_sgemm:
// logits = cembed . x_final (training/training_dynamic/train.m:490-491), dy = cembed^T . dlogits (:501-502),
// gcembed += dlogits . x_final^T (:507-508), and the dW products of each layer (:577-581, :613, :681-685).
//
// Large products go through the bfloat16 matrix instruction, each fp32 value as a sum of three (gemm_split.h); the kernel
// in this file takes the others.
//
// fp32 products on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: fp32 products and sums, 157 TFLOP/s on the
// chip).  An instruction takes 32 cycles of its SIMD for two registers of operands, so neither LDS nor memory is close to
// its limit and what counts is that every SIMD has an instruction to issue all the time: tiles that divide the output
// evenly over the compute units, several waves per SIMD, and K slices where the output alone has too few tiles.
// Measured against the library product that stood here before, [24573][1024] . [1024][256] and its two gradients:
// 109 us against 121, 118 against 144, 129 against 271 (70 -> 108 TFLOP/s over the three); 4096 x 4096 x 4096: 123
// TFLOP/s.  What is missing to 154, the rate of the instructions alone, goes to the LDS writes (a loop of instructions,
// fragment reads and barriers runs at 150, with the writes at 145) and to loads that have not arrived (134).
//
// A workgroup of four waves owns a BM x BN tile and walks K in steps of 16 through two LDS buffers (the next step's
// operands are fetched into registers while the current one is multiplied).  An operand tile lies in LDS as it lies in
// memory, so all four transpose cases load 128 bits per lane and transpose nothing:
//   K contiguous: [row][16 + 4], a lane reads four consecutive k of its row (128 bits, pitch 20: no bank conflicts);
//   K strided:    [16][BX + 4], a lane reads one element per k (the quarters of a wave read rows four apart, which the
//                 pitch puts into different quarters of the banks).
// The instruction takes k from the lane's quarter; which k that is may be chosen as long as both operands agree: of the
// four instructions of a step, number s multiplies k = s, 4 + s, 8 + s and 12 + s.
#include "tile.h"

#include <type_traits>

namespace {

constexpr int GK = 16;                 // K per step
constexpr int G_THREADS = 256;

// One operand tile of BX rows (of M or N) by GK: global -> registers -> LDS -> fragments.
// KC: k is the contiguous index of the operand in memory.
template <int BX, bool KC>
struct Operand {
    static constexpr int PITCH = KC ? GK + 4 : BX + 4;
    static constexpr int FLOATS = KC ? BX * PITCH : GK * PITCH;
    static constexpr int NV = BX * GK / 4 / G_THREADS;      // 128-bit pieces per thread
    static_assert(BX * GK % (4 * G_THREADS) == 0, "a tile is a whole number of pieces per thread");
    const float *src[NV];       // this thread's pieces of the step at hand
    size_t ahead;               // floats from one step to the next
    int left;                   // KC: unused; otherwise columns from the first piece to the end of the row
    v4f r[NV];

    static __device__ __forceinline__ void place(int i, int &x, int &k) {
        const int v = threadIdx.x + i * G_THREADS;
        if constexpr (KC) { x = v / (GK / 4); k = v % (GK / 4) * 4; }
        else { k = v / (BX / 4); x = v % (BX / 4) * 4; }
    }
    // rows x0 .. of X.  Rows past the end are read from the last one (K contiguous) or not at all; what they multiply is
    // never stored.
    __device__ __forceinline__ void start(const float *__restrict__ p, int ld, int x0, int X, int k0) {
        int x, k;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            place(i, x, k);
            src[i] = KC ? p + (size_t)min(x0 + x, X - 1) * ld + (k0 + k) : p + (size_t)(k0 + k) * ld + (x0 + x);
        }
        place(0, x, k);
        left = X - (x0 + x);
        ahead = KC ? (size_t)GK : (size_t)GK * ld;
    }
    // the pieces of a whole step; edge: the tile hangs over the end of the rows (the same for the whole workgroup)
    __device__ __forceinline__ void fetch(bool edge) {
#pragma unroll
        for (int i = 0; i < NV; i++) {
            if (KC || !edge || left >= 4) {
                r[i] = ld4(src[i]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) r[i][j] = j < left ? src[i][j] : 0.f;
            }
            src[i] += ahead;
        }
    }
    // the pieces of a step of which only n < GK values of k exist
    __device__ __forceinline__ void fetch_tail(int n) {
#pragma unroll
        for (int i = 0; i < NV; i++) {
            int x, k;
            place(i, x, k);
#pragma unroll
            for (int j = 0; j < 4; j++) r[i][j] = (KC ? k + j < n : k < n && j < left) ? src[i][j] : 0.f;
        }
    }
    __device__ __forceinline__ void put(float *lds) const {
#pragma unroll
        for (int i = 0; i < NV; i++) {
            int x, k;
            place(i, x, k);
            *reinterpret_cast<v4f *>(lds + (KC ? x * PITCH + k : k * PITCH + x)) = r[i];
        }
    }
    // the four values of row x (of this lane) for the steps of group g: k = 16g + 4*quarter + s
    static __device__ __forceinline__ v4f frag(const float *lds, int x, int g, int quarter) {
        if constexpr (KC) {
            return *reinterpret_cast<const v4f *>(lds + x * PITCH + 16 * g + 4 * quarter);
        } else {
            v4f f;
#pragma unroll
            for (int s = 0; s < 4; s++) f[s] = lds[(16 * g + 4 * quarter + s) * PITCH + x];
            return f;
        }
    }
};

// C = alpha * op(A) . op(B) + beta * C for one K slice; part != NULL: the bare product of the slice goes to part[slice].
// WM x WN: the tile of a wave.  Workgroup order: the tiles of one block of rows one after the other (their rows of A then
// come from one XCD's L2), slices outermost.
template <int BM, int BN, int WM, int WN, bool TA, bool TB>
__global__ __launch_bounds__(G_THREADS) void sgemm_kernel(const float *__restrict__ A, int lda, const float *__restrict__ B,
                                                          int ldb, float *C, int ldc, int M, int N, int K, int k_slice,
                                                          int tiles_n, int tiles, float alpha, float beta,
                                                          float *__restrict__ part) {
    typedef Operand<BM, !TA> OpA;
    typedef Operand<BN, TB> OpB;
    constexpr int FM = WM / 16, FN = WN / 16;
    constexpr bool EARLY_C = FM * FN <= 4;      // few enough values of C to hold them through the loop
    static_assert((BM / WM) * (BN / WN) == G_THREADS / 64, "four waves cover the tile");
    __shared__ __align__(16) float lds[2][OpA::FLOATS + OpB::FLOATS];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int slice = logical / tiles, tile = logical - slice * tiles;
    const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * BN;
    const int k_beg = slice * k_slice, k_end = min(K, k_beg + k_slice);
    const int steps = (k_end - k_beg) / GK, rest = (k_end - k_beg) % GK;
    const bool edge_m = m0 + BM > M, edge_n = n0 + BN > N;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;
    const int wm = wave / (BN / WN) * WM, wn = wave % (BN / WN) * WN;

    v4f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][j][e] = 0.f;

    // register e of a lane: row 4*quarter + e, column li of the 16 x 16 block
    float *out = part ? part + (size_t)slice * M * N : C;
    const int ldo = part ? N : ldc;
    float c[EARLY_C ? FM : 1][FN][4];
    auto each = [&](int i, auto f) {
        const int mb = m0 + wm + 16 * i + 4 * quarter;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const int n = n0 + wn + 16 * j + li;
                if (n < N && mb + e < M) f(c[EARLY_C ? i : 0][j][e], out[(size_t)(mb + e) * ldo + n]);
            }
    };
    const bool read = !part && beta != 0.f;           // beta == 0 does not read C (cblas semantics)
    if (EARLY_C && read) {
#pragma unroll
        for (int i = 0; i < FM; i++) each(i, [&](float &x, float &o) { x = o; });
    }

    OpA oa;
    OpB ob;
    oa.start(A, lda, m0, M, k_beg);
    ob.start(B, ldb, n0, N, k_beg);
    auto fetch = [&](int t) {
        if (t < steps) { oa.fetch(edge_m); ob.fetch(edge_n); }
        else { oa.fetch_tail(rest); ob.fetch_tail(rest); }
    };
    auto put = [&](int buf) { oa.put(lds[buf]); ob.put(lds[buf] + OpA::FLOATS); };
    const int all = steps + (rest > 0);
    // The fragments of a step are one set of registers; the next step's are asked for behind the barrier that follows the
    // next tile's way into LDS, with half a step of instructions still to issue.  (With everything at the end of the step
    // the waves of a SIMD reached their waits together: 110 TFLOP/s at 4096 x 4096 x 4096.)  Every buffer is read before
    // the barrier of its own step and written behind it.
    v4f a[2][FM], b[2][FN];
    auto frags = [&](int t, int g, int set) {
        const float *la = lds[t & 1], *lb = lds[t & 1] + OpA::FLOATS;
#pragma unroll
        for (int i = 0; i < FM; i++) a[set][i] = OpA::frag(la, wm + 16 * i + li, g, quarter);
#pragma unroll
        for (int j = 0; j < FN; j++) b[set][j] = OpB::frag(lb, wn + 16 * j + li, g, quarter);
    };
    auto multiply = [&](int set, int s0, int s1) {
#pragma unroll
        for (int s = s0; s < s1; s++)
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[set][i][s], b[set][j][s], acc[i][j], 0, 0, 0);
    };
    fetch(0);
    put(0);
    if (all > 1) fetch(1);
    __syncthreads();
    frags(0, 0, 0);
    for (int t = 0; t < all; t += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (t + u < all) {
                const bool more = t + u + 1 < all;
                multiply(u, 0, 2);
                __builtin_amdgcn_sched_barrier(0);
                if (more) {
                    put((u + 1) & 1);
                    if (t + u + 2 < all) fetch(t + u + 2);
                }
                __syncthreads();
                if (more) frags(u + 1, 0, (u + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(u, 2, 4);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < FM; i++) {
        if (!EARLY_C && read) each(i, [&](float &x, float &o) { x = o; });
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float &x = c[EARLY_C ? i : 0][j][e];
                const float p = part ? acc[i][j][e] : acc[i][j][e] * alpha;
                x = read ? p + beta * x : p;
            }
        each(i, [&](float &x, float &o) { o = x; });
    }
}

#include "gemm_split.h"

// C = alpha * sum_s part[s] + beta * C, s ascending
__global__ __launch_bounds__(256) void slice_sum_kernel(float *C, int ldc, const float *__restrict__ part, int slices, int M,
                                                        int N, float alpha, float beta) {
    const size_t n = (size_t)M * N, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float acc = 0.f;
#pragma unroll 4
    for (int s = 0; s < slices; s++) acc += __builtin_nontemporal_load(part + (size_t)s * n + i);
    float *o = C + i / N * (size_t)ldc + i % N;
    *o = alpha * acc + (beta != 0.f ? beta * *o : 0.f);
}

// 0 / 111 (CblasNoTrans) -> false, 1 / 112 (CblasTrans) -> true, anything else -> -1
int trans_flag(int t) {
    if (t == 0 || t == 111) return 0;
    if (t == 1 || t == 112) return 1;
    return -1;
}

struct GemmPlan {
    int split, bm, bn, slices, k_slice;      // split: the kernel of gemm_split.h
};

// The kernel, tile and number of K slices with the least estimated time.
// Split kernel: a workgroup has a compute unit to itself and takes 2.5 us a step of 32 and 4 us around them (4 more where
// it reads C).  fp32 kernel: a compute unit multiplies 0.48 MFLOP a microsecond (123 TFLOP/s on the chip, measured at
// 4096^3 with every tile size) when two or more workgroups share it; with one, whose waves wait at their barriers, three
// quarters of that.  Slices cost their partial products' way through memory and a launch; they pay where the output has
// few tiles.  Measured, split kernel against fp32 kernel, us, and relative error of either against 64 bits:
//   [24573][1024] . [1024][256]      86 / 109    5.0e-7 / 5.7e-7    (the library that stood here first: 121, 5.7e-7)
//   [1024][24573] . [24573][256]     80 / 118    5.0e-7 / 10e-7     (144, 5.2e-7)
//   [24573][256] . [256][1024] +=    90 / 129    2.6e-7 / 2.9e-7    (271, 2.9e-7)
//   [9001][768] . [768][197]         39 / 49     2.6e-7 / 5.0e-7    [768][9001] . [9001][197]  34 / 44   2.8e-7 / 4.3e-7
//   [768][768] . [768][256]          18 / 11     2.0e-7 / 2.3e-7    [2000][32] . [32][768]     7.6 / 5   1.2e-7 / 1.0e-7
// The large tiles lose where the output has few of them, and the estimate leaves those to the fp32 kernel, of whose tiles
// only the smallest holds the old values of C through its loop.
GemmPlan plan_gemm(int M, int N, int K, bool reads_c, int lda, int ldb) {
    const int cus = g_ctx.num_cu > 0 ? g_ctx.num_cu : 256;
    struct Tile { int split, bm, bn; };
    const Tile tile[5] = {{0, 128, 64}, {0, 64, 128}, {0, 64, 64}, {1, 128, 256}, {1, 256, 128}};
    GemmPlan best = {0, 64, 64, 1, K};
    double best_us = -1.0;
    const bool can = lda < (1 << 22) && ldb < (1 << 22);        // (32-bit offsets of the lanes)
    for (const Tile &t : tile) {
        if (t.split ? g_ctx.gemm_split < 0 || !can : g_ctx.gemm_split > 0 && can) continue;
        if (t.split && g_ctx.gemm_split > 0 && t.bm != 128 * g_ctx.gemm_split) continue;
        const int step = t.split ? SK : GK;
        const double tiles = (double)ceil_div((size_t)M, (size_t)t.bm) * (double)ceil_div((size_t)N, (size_t)t.bn);
        for (int want = 1; want <= 64; want++) {
            if (g_ctx.gemm_splitk && want != (K >= 2 * g_ctx.gemm_splitk ? g_ctx.gemm_splitk : 1)) continue;
            const int k_slice = (int)ceil_div(ceil_div((size_t)K, (size_t)want), (size_t)step) * step;
            const int slices = (int)ceil_div((size_t)K, (size_t)k_slice);
            if (want > 1 && !g_ctx.gemm_splitk && (k_slice < 128 || (double)slices * M * N > 64e6)) break;
            const double per_cu = tiles * slices / cus;
            const double rounds = per_cu <= 1.0 ? 1.0 : (double)(long)(per_cu + 0.999999);
            const double mflop = (double)t.bm * t.bn * k_slice * 2.0e-6;
            double us;
            if (t.split) us = rounds * (4.0 + 2.5 * (k_slice / SK)) + (reads_c && slices == 1 ? rounds * 4.0 : 0.0);
            else us = rounds * mflop / 0.48 * (per_cu <= 1.0 ? 1.33 : 1.0);
            if (!t.split && reads_c && slices == 1 && t.bm * t.bn > 64 * 64) us *= 1.05;
            if (slices > 1) us += 5.0 + (double)slices * M * N * 8.0 / 5e6;
            if (best_us < 0.0 || us < best_us) { best_us = us; best = GemmPlan{t.split, t.bm, t.bn, slices, k_slice}; }
        }
    }
    return best;
}

// The product within the limits of one launch: M, K <= 2^30, fewer than 2^24 workgroups (the caller cuts larger ones).
int sgemm_piece(int ta, int tb, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta,
                float *C, int ldc) {
    const GemmPlan p = plan_gemm(M, N, K, beta != 0.f, lda, ldb);
    float *part = nullptr;
    if (p.slices > 1) {
        part = (float *)mi355_ws((size_t)p.slices * M * N * sizeof(float));
        if (!part) return -1;
    }
    const int tiles_n = (int)ceil_div((size_t)N, (size_t)p.bn), tiles = (int)ceil_div((size_t)M, (size_t)p.bm) * tiles_n;
    // alpha == 0 reads neither operand (cblas semantics): a product over nothing
    const int k_all = alpha != 0.f ? K : 0;
    auto launch = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)tiles * p.slices), dim3(threads), 0, g_ctx.stream, A, lda, B, ldb, C, ldc, M, N,
                           k_all, p.k_slice, tiles_n, tiles, alpha, beta, part);
    };
#define GEMM_CASE(BM, BN, WM, WN)                                                                                     \
    case (BM) * 1000 + (BN):                                                                                          \
        if (!ta && !tb) launch(sgemm_kernel<BM, BN, WM, WN, false, false>, G_THREADS);                                \
        else if (!ta) launch(sgemm_kernel<BM, BN, WM, WN, false, true>, G_THREADS);                                   \
        else if (!tb) launch(sgemm_kernel<BM, BN, WM, WN, true, false>, G_THREADS);                                   \
        else launch(sgemm_kernel<BM, BN, WM, WN, true, true>, G_THREADS);                                             \
        break;
#define SPLIT_CASE(BM, BN)                                                                                            \
    case (BM) * 1000 + (BN):                                                                                          \
        if (!ta && !tb) launch(sgemm_split_kernel<BM, BN, false, false>, S_THREADS);                              \
        else if (!ta) launch(sgemm_split_kernel<BM, BN, false, true>, S_THREADS);                                 \
        else if (!tb) launch(sgemm_split_kernel<BM, BN, true, false>, S_THREADS);                                 \
        else launch(sgemm_split_kernel<BM, BN, true, true>, S_THREADS);                                           \
        break;
    switch (p.bm * 1000 + p.bn) {
        GEMM_CASE(64, 128, 32, 64)
        GEMM_CASE(128, 64, 64, 32)
        GEMM_CASE(64, 64, 32, 32)
        SPLIT_CASE(128, 256)
        SPLIT_CASE(256, 128)
        default: return mi355_fail("sgemm: no kernel for a tile of %d x %d", p.bm, p.bn);
    }
#undef GEMM_CASE
#undef SPLIT_CASE
    LAUNCH_OK("sgemm");
    if (part) {
        hipLaunchKernelGGL(slice_sum_kernel, dim3((unsigned)ceil_div((size_t)M * N, 256)), dim3(256), 0, g_ctx.stream, C, ldc,
                           part, p.slices, M, N, alpha, beta);
        LAUNCH_OK("sgemm slice sum");
    }
    return 0;
}

}   // namespace

MI355_API int mi355_sgemm_dev(int trans_a, int trans_b, int M, int N, int K, float alpha, const float *A, int lda,
                              const float *B, int ldb, float beta, float *C, int ldc) {
    if (!mi355_ready("sgemm")) return -1;
    if (!mi355_outside_capture("sgemm (its K slices may need workspace)")) return -1;
    if (!A || !B || !C) return mi355_fail("sgemm: NULL pointer");
    const int ta = trans_flag(trans_a), tb = trans_flag(trans_b);
    if (ta < 0 || tb < 0) return mi355_fail("sgemm: transpose flags must be 0/1 (or CblasNoTrans/CblasTrans)");
    if (M <= 0 || N <= 0 || K <= 0) return mi355_fail("sgemm: bad shape M=%d N=%d K=%d", M, N, K);
    // row-major leading dimensions: A is M x K (or K x M when transposed), B is K x N (or N x K), C is M x N
    if (lda < (ta ? M : K) || ldb < (tb ? K : N) || ldc < N)
        return mi355_fail("sgemm: leading dimension too small (lda=%d ldb=%d ldc=%d)", lda, ldb, ldc);
    // Pieces of what a launch can number and 32-bit arithmetic on rows and k can hold: 2^30 values of k, 2^26 rows, and as many
    // columns as make 2^23 tiles of 64 x 64.  All but thin or long products beyond a billion rows or columns are one piece.
    constexpr int KC = 1 << 30, MC = 1 << 26;
    const int mc = M < MC ? M : MC;
    const size_t tiles_n = ((size_t)1 << 23) / ceil_div((size_t)mc, 64);
    const int nc = (size_t)N > 64 * tiles_n ? (int)(64 * tiles_n) : N;
    for (long long m = 0; m < M; m += mc)
        for (long long n = 0; n < N; n += nc)
            for (long long k = 0; k < K; k += KC) {
                const int pm = (int)(M - m < mc ? M - m : mc), pn = (int)(N - n < nc ? N - n : nc);
                const int pk = (int)(K - k < KC ? K - k : KC);
                if (sgemm_piece(ta, tb, pm, pn, pk, alpha, A + (ta ? m + k * lda : m * lda + k), lda,
                                B + (tb ? n * ldb + k : n + k * ldb), ldb, k == 0 ? beta : 1.0f, C + m * ldc + n, ldc))
                    return -1;
                if (alpha == 0.f) break;
            }
    return 0;
}
