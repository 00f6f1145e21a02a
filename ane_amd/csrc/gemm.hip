// gemm.hip — the loops' cblas_sgemm(CblasRowMajor, ...) calls on device memory.
//
// The dynamic loop runs the classifier and every weight-gradient product on the CPU through cblas_sgemm:
// logits = cembed . x_final (training/training_dynamic/train.m:490-491), dy = cembed^T . dlogits (:501-502),
// gcembed += dlogits . x_final^T (:507-508), and the dW products of each layer (:577-581, :613, :681-685).
//
// Large products and many of middle size go through the bfloat16 matrix instruction, each fp32 value as a sum of three
// (gemm_split.h; gemm_planes.h where one operand is small enough to be split ahead); the kernel in this file takes the others
// (plan_gemm).
//
// fp32 products on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: fp32 products and sums, 157 TFLOP/s on the
// chip).  An instruction takes 32 cycles of its SIMD for two registers of operands, so neither LDS nor memory is close to
// its limit and what counts is that every SIMD has an instruction to issue all the time: tiles that divide the output
// evenly over the compute units, several waves per SIMD, and K slices where the output alone has too few tiles.
// 4096 x 4096 x 4096 runs at 120 TFLOP/s; what is missing to 154, the rate of the instructions alone, goes to the LDS writes
// (a loop of instructions, fragment reads and barriers runs at 150, with the writes at 145) and to loads that have not
// arrived (134).  A wave takes 32 x 32 of the output; four waves with 64 x 64 where every compute unit has several workgroups.
// Smaller outputs leave a compute unit with one, whose four waves wait at its barriers together, so there eight waves share
// a tile of 64 x 64, 64 x 32 or 32 x 64, in two or four groups with their own part of k:
// 2048 x 256 x 768 17 us with four waves, 10.8 with eight (the library that stood here before: 14),
// [2048][256] . [256][768] += 13.2 and 11.4 (11); sums of a half or a quarter of the terms round less (errors at plan_gemm).
//
// A workgroup owns a BM x BN tile and walks K in steps of 16 per group through two LDS buffers; the next step is on its way to
// registers.  Where there are groups a wave's fragments of a step are one set of registers, so that three workgroups fit a
// compute unit (62 to 67 registers; with two sets 90, two workgroups, and 12.2 us for the 11.4 above).  Larger tiles (128 x 64
// with 48 accumulators, one or two steps ahead) are nowhere faster.  An operand tile lies in LDS as it lies in
// memory, so all four transpose cases load 128 bits per lane and transpose nothing:
//   K contiguous: [row][K + 4], a lane reads four consecutive k of its row (128 bits; pitches of 20, 36 and 68 floats have no
//                 bank conflicts);
//   K strided:    [K][BX + 4], a lane reads one element per k (the quarters of a wave read rows four apart, which the
//                 pitch puts into different quarters of the banks).
// The instruction takes k from the lane's quarter; which k that is may be chosen as long as both operands agree: of the
// four instructions of a group's step, number s multiplies k = s, 4 + s, 8 + s and 12 + s of its sixteen.
#include "tile.h"

#include <algorithm>
#include <type_traits>

void mi355_free_planes(void);

namespace {

constexpr int GK = 16;                 // K per step and group of waves

// One operand tile of BX rows (of M or N) by K values of k, by THREADS threads: global -> registers -> LDS -> fragments.
// KC: k is the contiguous index of the operand in memory.
template <int BX, bool KC, int K, int THREADS>
struct Operand {
    static constexpr int PITCH = KC ? K + 4 : BX + 4;
    static constexpr int FLOATS = KC ? BX * PITCH : K * PITCH;
    static constexpr int NV = BX * K / 4 / THREADS;         // 128-bit pieces per thread
    static_assert(BX * K % (4 * THREADS) == 0 && THREADS % (BX / 4) == 0, "a tile is a whole number of pieces per thread");
    const float *src[NV];       // this thread's pieces of the step at hand
    size_t ahead;               // floats from one step to the next
    int left;                   // KC: unused; otherwise columns from the first piece to the end of the row
    v4f r[NV];

    static __device__ __forceinline__ void place(int i, int &x, int &k) {
        const int v = threadIdx.x + i * THREADS;
        if constexpr (KC) { x = v / (K / 4); k = v % (K / 4) * 4; }
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
        ahead = KC ? (size_t)K : (size_t)K * ld;
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
    // the pieces of a step of which only n < K values of k exist
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
    // the four values of row x (of this lane) for group g of waves: k = 16g + 4*quarter + s
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

template <int BM, int BN, int WM, int WN, int KS>
struct GemmShape {
    static constexpr int WAVES = (BM / WM) * (BN / WN);      // of a group
    static constexpr int THREADS = 64 * WAVES * KS;
};

// C = alpha * op(A) . op(B) + beta * C for one K slice; part != NULL: the bare product of the slice goes to part[slice].
// WM x WN: the tile of a wave.  KS groups of waves compute the same BM x BN tile, each over its sixteen of the 16 * KS values
// of k in a step; at the end each group adds up its share of the tile, in group order.  Workgroup order: the tiles of one
// block of rows one after the other (their rows of A then come from one XCD's L2), slices outermost.
template <int BM, int BN, int WM, int WN, int KS, bool TA, bool TB>
__global__ __launch_bounds__(64 * KS * (BM / WM) * (BN / WN), KS > 1 ? 6 : 1) void sgemm_kernel(
    const float *__restrict__ A, int lda, const float *__restrict__ B, int ldb, float *C, int ldc, int M, int N, int K,
    int k_slice, int tiles_n, int tiles, float alpha, float beta, float *__restrict__ part) {
    typedef GemmShape<BM, BN, WM, WN, KS> Shape;
    constexpr int STEP = GK * KS;
    typedef Operand<BM, !TA, STEP, Shape::THREADS> OpA;
    typedef Operand<BN, TB, STEP, Shape::THREADS> OpB;
    constexpr int FM = WM / 16, FN = WN / 16;
    constexpr int OWN = FM * FN / KS;           // fragments that a group finishes
    static_assert(FM * FN % KS == 0, "the groups share the fragments evenly");
    constexpr int BUF = OpA::FLOATS + OpB::FLOATS;
    __shared__ __align__(16) float lds[2][BUF];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int slice = logical / tiles, tile = logical - slice * tiles;
    const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * BN;
    const int k_beg = slice * k_slice, k_end = min(K, k_beg + k_slice);
    const int steps = (k_end - k_beg) / STEP, rest = (k_end - k_beg) % STEP;
    const bool edge_m = m0 + BM > M, edge_n = n0 + BN > N;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;
    const int group = wave / Shape::WAVES, ww = wave % Shape::WAVES;
    const int wm = ww / (BN / WN) * WM, wn = ww % (BN / WN) * WN;

    v4f acc[FM * FN];
#pragma unroll
    for (int f = 0; f < FM * FN; f++) acc[f] = v4f{0.f, 0.f, 0.f, 0.f};

    // register e of a lane of fragment f: row 4*quarter + e, column li of its 16 x 16 block
    float *out = part ? part + (size_t)slice * M * N : C;
    const int ldo = part ? N : ldc;
    v4f c[OWN];                                       // held through the loop
    auto each = [&](auto fn) {
        auto one = [&](int i, int e, int j) {
            const int m = m0 + wm + 16 * i + 4 * quarter + e, n = n0 + wn + 16 * j + li;
            if (n < N && m < M) fn(i * FN + j, e, out[(size_t)m * ldo + n]);
        };
        if constexpr (KS == 1) {                      // row by row, so that the pieces of a line follow one another
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int j = 0; j < FN; j++) one(i, e, j);
        } else {
#pragma unroll
            for (int f = 0; f < FM * FN; f++)
                if (f / OWN == group) {
#pragma unroll
                    for (int e = 0; e < 4; e++) one(f / FN, e, f % FN);
                }
        }
    };
    const bool read = !part && beta != 0.f;           // beta == 0 does not read C (cblas semantics)
    if (read) each([&](int f, int e, float &o) { c[f % OWN][e] = o; });

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
    // With one group the next step's fragments are asked for behind the barrier that follows the next tile's way into LDS,
    // with half a step of instructions still to issue.  (With everything at the end of the step the waves of a SIMD reached
    // their waits together: 110 TFLOP/s at 4096 x 4096 x 4096.)  Every buffer is read before the barrier of its own step and
    // written behind it.
    constexpr int FS = KS == 1 ? 2 : 1;
    v4f a[FS][FM], b[FS][FN];
    auto frags = [&](int t, int set) {
        const float *la = lds[t & 1], *lb = lds[t & 1] + OpA::FLOATS;
#pragma unroll
        for (int i = 0; i < FM; i++) a[set][i] = OpA::frag(la, wm + 16 * i + li, group, quarter);
#pragma unroll
        for (int j = 0; j < FN; j++) b[set][j] = OpB::frag(lb, wn + 16 * j + li, group, quarter);
    };
    auto multiply = [&](int set, int s0, int s1) {
#pragma unroll
        for (int s = s0; s < s1; s++)
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++)
                    acc[i * FN + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[set][i][s], b[set][j][s], acc[i * FN + j], 0, 0, 0);
    };
    fetch(0);
    put(0);
    if (all > 1) fetch(1);
    __syncthreads();
    frags(0, 0);
    for (int t = 0; t < all; t += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (t + u < all) {
                const bool more = t + u + 1 < all;
                multiply(u % FS, 0, FS == 1 ? 4 : 2);
                __builtin_amdgcn_sched_barrier(0);
                if (more) {
                    put((u + 1) & 1);
                    if (t + u + 2 < all) fetch(t + u + 2);
                }
                __syncthreads();
                if (more) frags(u + 1, (u + 1) % FS);
                __builtin_amdgcn_sched_barrier(0);
                if (FS > 1) multiply(u % FS, 2, 4);
            }
        }
    }
    if constexpr (KS > 1) {
        // every group's sums of the fragments that others finish: [fragment][group][wave of a group][lane]
        static_assert(FM * FN * KS * Shape::WAVES * 256 <= 2 * BUF, "the sums fit the buffers");
        v4f *x = reinterpret_cast<v4f *>(&lds[0][0]);
        auto at = [&](int f, int g) { return ((f * KS + g) * Shape::WAVES + ww) * 64 + lane; };
        __syncthreads();
#pragma unroll
        for (int f = 0; f < FM * FN; f++)
            if (f / OWN != group) x[at(f, group)] = acc[f];
        __syncthreads();
#pragma unroll
        for (int f = 0; f < FM * FN; f++)
            if (f / OWN == group) {
                v4f s = group == 0 ? acc[f] : x[at(f, 0)];
#pragma unroll
                for (int g = 1; g < KS; g++) s += g == group ? acc[f] : x[at(f, g)];
                acc[f] = s;
            }
    }
    each([&](int f, int e, float &o) {
        const float p = part ? acc[f][e] : acc[f][e] * alpha;
        o = read ? p + beta * c[f % OWN][e] : p;
    });
}

#include "gemm_split.h"
#include "gemm_planes.h"

// C = alpha * sum_s part[s] + beta * C.  GROUPS threads to an element: thread g adds the slices g, g + GROUPS, ... in order,
// then the groups' sums are added in order.  One thread to an element waits for slices / 4 trips to memory one after the
// other (a product of 1 x 1 x 1000000 in 256 slices: 15 us of its 49).
template <int GROUPS>
__global__ __launch_bounds__(256) void slice_sum_kernel(float *C, int ldc, const float *__restrict__ part, int slices, int M,
                                                        int N, float alpha, float beta) {
    constexpr int EL = 256 / GROUPS;
    __shared__ float sum[GROUPS][EL];
    const size_t n = (size_t)M * N, i = (size_t)blockIdx.x * EL + threadIdx.x % EL;
    const int g = threadIdx.x / EL;
    float acc = 0.f;
    if (i < n) {
#pragma unroll 4
        for (int s = g; s < slices; s += GROUPS) acc += __builtin_nontemporal_load(part + (size_t)s * n + i);
    }
    if constexpr (GROUPS > 1) {
        sum[g][threadIdx.x % EL] = acc;
        __syncthreads();
        if (g > 0) return;
#pragma unroll
        for (int k = 1; k < GROUPS; k++) acc += sum[k][threadIdx.x];
    }
    if (i >= n) return;
    float *o = C + i / N * (size_t)ldc + i % N;
    *o = alpha * acc + (beta != 0.f ? beta * *o : 0.f);
}

// 0 / 111 (CblasNoTrans) -> false, 1 / 112 (CblasTrans) -> true, anything else -> -1
int trans_flag(int t) {
    if (t == 0 || t == 111) return 0;
    if (t == 1 || t == 112) return 1;
    return -1;
}

// split: the bfloat16 instruction, 1 with both operands split by every tile (gemm_split.h), 2 and 3 with B split ahead
// (gemm_planes.h: sgemm_planes_kernel, sgemm_rows_kernel); groups of waves; ranges of columns (3)
struct GemmPlan {
    int split, groups, bm, bn, slices, k_slice, ranges;
};
constexpr int gemm_key(int split, int groups, int bm, int bn) { return ((split * 10 + groups) * 1000 + bm) * 1000 + bn; }

// A kernel and what it takes, in us: a step of `step` values of k where one workgroup has a compute unit to itself, where
// several share it (of each), and what surrounds the steps, once for every `resident` workgroups of a compute unit.
struct GemmKernel {
    int split, groups, bm, bn, step, resident;
    double alone, shared, fixed;
};
constexpr GemmKernel GEMM_KERNELS[] = {
    {0, 1, 64, 64, 16, 4, 0.41, 0.30, 0.14}, {0, 2, 64, 64, 32, 3, 0.48, 0.49, 1.7},
    {0, 4, 64, 32, 64, 3, 0.66, 0.66, 0.27}, {0, 4, 32, 64, 64, 3, 0.66, 0.66, 0.27},
    {1, 1, 128, 256, 32, 1, 2.3, 2.6, 4.2},  {1, 1, 256, 128, 32, 1, 2.3, 2.6, 4.2},
    {1, 1, 64, 64, 32, 3, 0.93, 0.43, 2.1},  {1, 2, 64, 64, 64, 1, 0.86, 0.86, 2.7},
    {2, 1, 96, 256, 64, 1, 3.7, 3.7, 4.4},   {2, 1, 64, 256, 64, 1, 2.6, 2.6, 4.4},
};
// The kernel and number of K slices with the least estimated time: a launch, the longer of the work of the busiest compute
// unit and the bytes from memory at 5.6 TB/s or from the L2s at 21, and a quarter of the shorter one, which do not overlap
// better than that.  fp32 operands whose k is strided take a sixth longer (their fragments are read a float at a time).
// Slices cost a launch and the way of their partial products through memory, an operand split ahead a launch and its way at
// the rate of the last-level cache.  The numbers are fitted to 210 products of every transpose case (vocabularies of 2000 to
// 24573 rows by 32 to 512 columns, the weight gradients of a layer, squares, thin and long ones) in every kernel and number of
// slices, those of gemm_planes.h to 153 of them: what is chosen takes 0.7 % more than the best on the average and 14 % at worst;
// tiles of 128 x 64 and 64 x 128 were never the best and are gone.  On 380 other products, odd sizes among them, whose operands
// no cache holds, it takes 2.2 % more than the best of the kernels on the average, 5 % more in 57 and 58 % more at worst ([1000][768]^T
// . [1000][500], fp32 32 x 64 27.9, split 64 x 64 in two groups 17.7).
// Measured on operands that the caches hold, us; the chosen kernel first (in brackets the library that stood here before).  Where
// they do not, the same ones are ahead: [24573][1024] . [1024][256] 72, split 256 x 128 91; [24573][256] . [256][1024] += 82, 105;
// [32000][256] . [256][768] += 90, 104; [32000][768] . [768][256] 75, planes 64 x 256 81; [768][32000] . [32000][256] 82, planes 87;
// [14000][768] . [768][256] 43, 52; [14000][256] . [256][768] += 45, split 64 x 64 58; [24573][64] . [64][1024] += 58, fp32 66.
//   [24573][1024] . [1024][256]        planes 96 x 256 71, split 256 x 128 90, 64 x 64 100, fp32 124
//   [24573][256] . [256][1024] +=      rows of 96 68, split 128 x 256 94, 64 x 64 107, fp32 123
//   [32000][256] . [256][768] +=       rows of 64 73, of 96 82, split 128 x 256 90, fp32 121                   (112)
//   [32000][768] . [768][256]          split 128 x 256 68, planes 64 x 256 78, 96 x 256 92, fp32 115           (105)
//   [768][32000] . [32000][256]        split 128 x 256 in 32 slices 80, planes 96 x 256 84, fp32 120           (328)
//   [9001][768] . [768][197]           split 64 x 64 35, planes 64 x 256 37, fp32 64 x 32 41                   (42)
//   [14000][768] . [768][256]          planes 64 x 256 39, split 256 x 128 48, 64 x 64 52, fp32 61
//   [14000][256] . [256][768] +=       rows of 64 37, of 96 43, split 64 x 64 51, fp32 58
//   [24573][64] . [64][1024] +=        rows of 96 41, fp32 64 x 64 55, split 128 x 256 56, 64 x 64 59          (42)
//   [2048][256] . [256][768] +=        fp32 32 x 64 11.8, 64 x 64 13.1, split 64 x 64 13.6, rows of 64 20      (10.9)
//   [3072][256] . [256][1024] +=       split 64 x 64 18.0, fp32 64 x 64 20.1, rows of 64 24, split 128 x 256 27 (16.3)
//   [4096][1024] . [1024][3072]        planes 64 x 256 140, split 128 x 256 168, 64 x 64 181, fp32 228
//   [4096][4096] . [4096][4096]        split 128 x 256 691, planes 96 x 256 725, 64 x 256 760 (6.4 GB of planes from the L2s), fp32 1183
//   [256][4096] . [4096][256]          fp32 32 x 64 12.5, split 64 x 64 in two groups 15.6
//   [1024][1024] . [1024][1024]        split 64 x 64 in two groups 21.6, fp32 64 x 32 23.5, 64 x 64 23.7       (19.9)
//   [2048][768] . [768][256]           fp32 64 x 32 10.9, split 64 x 64 in two groups 15.4, fp32 64 x 64 17    (13.8)
//   [24573][1024] . [1024][1]          fp32 64 x 32 24.5, split 64 x 64 32, fp32 64 x 64 38                    (72)
//   [32][100000] . [100000][32]        fp32 32 x 64 in 256 slices 12.7                                         (28)
//   [1][1000000] . [1000000][1]        fp32 32 x 64 in 256 slices 45, all of it for one element of a tile      (32)
// Relative error against 64 bits (2-norms, normal operands):
//   K       fp32, one group     two / four groups      split 64 x 64  split 128 x 256  planes   rows     (library)
//   32           1.03e-7            0.8e-7 / 0.8e-7       0.39e-7        1.17e-7       0.4e-7   0.4e-7   1.03e-7
//   64           1.44e-7            1.1e-7 / 0.8e-7       0.50e-7        1.46e-7       0.53e-7  0.53e-7  1.44e-7
//   80           1.61e-7            1.2e-7 / 1.0e-7       0.54e-7        1.56e-7       0.55e-7  0.57e-7  1.61e-7
//   256          2.87e-7            2.1e-7 / 1.5e-7       0.93e-7        2.57e-7       0.69e-7  0.74e-7  2.87e-7 (2.06e-7 in slices)
//   1024         5.72e-7            4.1e-7 / 2.9e-7       1.86e-7        5.0e-7        0.97e-7     -     5.72e-7
// so the large split tiles, whose hh products and small ones share a sum, are not taken below K = 80.
// ahead: B may be split ahead (there is memory for its planes).
GemmPlan plan_gemm(int ta, int tb, int M, int N, int K, bool reads_c, int lda, int ldb, int ldc, bool ahead) {
    const int cus = g_ctx.num_cu > 0 ? g_ctx.num_cu : 256;
    GemmPlan best = {0, 1, 64, 64, 1, K, 1};
    double best_us = -1.0;
    const bool can = lda < (1 << 22) && ldb < (1 << 22);        // (32-bit offsets of the lanes)
    const int knob = can ? g_ctx.gemm_split : -1;
    const auto up = [](double x) { return (double)(long)(x + 0.999999); };
    const double planes = (double)plane_bytes(N, K);
    const bool planes_ok = can && ahead && planes <= (double)P_MAX_BYTES;
    const double split_us = 1.9 + (4.0 * N * K + planes) / 15.4e6;         // the launch that splits B
    const double c_times = reads_c ? 2 : 1;
    for (const GemmKernel &t : GEMM_KERNELS) {
        // as the knob numbers them
        const int id = !t.split ? -1 : t.split == 2 ? (t.bm == 96 ? 5 : 6) : t.bm == 64 ? 2 + t.groups : t.bm / 128;
        if (t.split == 2 && !planes_ok) continue;
        if (knob ? (knob < 0 ? t.split != 0 : id != knob) : t.split != 2 && t.bm * t.bn > 64 * 64 && K < 80) continue;
        const double tiles_m = (double)ceil_div((size_t)M, (size_t)t.bm), tiles_n = (double)ceil_div((size_t)N, (size_t)t.bn);
        const double slow = t.split ? 1.0 : 1.0 + 0.16 * ((ta ? 1 : 0) + (tb ? 0 : 1));
        // slices: a few, and what fills every compute unit once, twice and three times
        const auto fill = [&](int times) { return (int)std::max(1.0, std::min(256.0, times * cus / (tiles_m * tiles_n))); };
        for (int want : {1, 2, 3, 4, 6, 8, fill(1), fill(2), fill(3)}) {
            if (g_ctx.gemm_splitk) want = K >= 2 * g_ctx.gemm_splitk ? g_ctx.gemm_splitk : 1;
            const int steps = (int)ceil_div(ceil_div((size_t)K, (size_t)want), (size_t)t.step), k_slice = steps * t.step;
            const int slices = (int)ceil_div((size_t)K, (size_t)k_slice);
            const double out = (double)M * N;
            if (want > 1 && !g_ctx.gemm_splitk && (k_slice < 128 || slices * out > 64e6)) continue;
            const double n = up(tiles_m * tiles_n * slices / cus);                      // workgroups of the busiest compute unit
            const double work = steps * std::max(t.alone, n * t.shared) * slow + t.fixed * up(n / t.resident);
            const double hbm = 4.0 * ((double)M * K + out * (slices > 1 ? slices : c_times)) + (t.split == 2 ? planes : 4.0 * N * K);
            // (a value of B's planes has six bytes; these kernels ask for them and for A a step ahead, so half of it counts)
            const double l2 = t.split == 2 ? K * (2.0 * M * tiles_n + 3.0 * N * tiles_m) : 4.0 * K * (M * tiles_n + N * tiles_m);
            const double mem = std::max(hbm / 5.6e6, l2 / 21e6);
            double us = 3.4 + std::max(work, mem) + 0.23 * std::min(work, mem);
            if (slices > 1) us += 5.4 + slices * out * 4.0 / 5.6e6;
            if (t.split == 2) us += split_us;
            if (best_us < 0.0 || us < best_us) { best_us = us; best = GemmPlan{t.split, t.groups, t.bm, t.bn, slices, k_slice, 1}; }
        }
    }
    // Rows of A held whole, 96 or 64 of them: the columns dealt out over a few ranges, each with a workgroup of its own per block
    // of rows, where the blocks alone leave compute units idle.
    for (int fm : {6, 4}) {
        if (knob ? knob != (fm == 6 ? 7 : 8) : g_ctx.gemm_splitk > 1) continue;
        if (!planes_ok || plane_steps(K) > rows_steps(fm) || ldc >= (1 << 22)) continue;        // (32-bit offsets into C)
        const int units = (int)ceil_div((size_t)N, 32), waves = R_THREADS / 64;
        const double blocks = (double)ceil_div((size_t)M, 16 * (size_t)fm);
        for (int want = 1; want <= 8 && waves * (want - 1) < units; want++) {
            const int per = (int)ceil_div((size_t)units, (size_t)want), ranges = (int)ceil_div((size_t)units, (size_t)per);
            if (per > R_UNITS) continue;
            const double work = up(blocks * ranges / cus) * (5.5 + up((double)per / waves) * (0.55 + plane_steps(K) * fm * 0.357));
            const double mem = (4.0 * ((double)M * K * ranges + (double)M * N * c_times) + planes) / 5.6e6;
            const double us = 3.4 + split_us + std::max(work, mem) + 0.21 * std::min(work, mem);
            if (best_us < 0.0 || us < best_us) { best_us = us; best = GemmPlan{3, 1, 16 * fm, 32 * per, 1, K, ranges}; }
        }
    }
    return best;
}

// Where the planes of an operand lie: grow-only, at most P_MAX_BYTES and the flags, freed with the caches.  Not the workspace: a
// product is never recorded, so no graph holds this address and none goes stale when a product needs more of it.  NULL where
// there is no memory for it (the other kernels then take the product).
char *g_planes = nullptr;
size_t g_planes_bytes = 0;
char *plane_space(size_t bytes) {
    if (bytes <= g_planes_bytes) return g_planes;
    mi355_free_planes();
    const size_t want = (bytes + 0xFFFFF) & ~(size_t)0xFFFFF;   // 1 MiB granules
    void *p = nullptr;
    if (hipMalloc(&p, want) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    g_planes = (char *)p;
    g_planes_bytes = want;
    return g_planes;
}

// The product within the limits of one launch: M, N, K <= 2^30 and 2^21 tiles of 64 x 64 (the caller cuts larger ones).
int sgemm_piece(int ta, int tb, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta,
                float *C, int ldc) {
    // (alpha == 0 reads neither operand: nothing is split ahead)
    GemmPlan p = plan_gemm(ta, tb, M, N, K, beta != 0.f, lda, ldb, ldc, alpha != 0.f);
    char *planes = nullptr;
    if (p.split >= 2 && !(planes = plane_space(plane_bytes(N, K)))) p = plan_gemm(ta, tb, M, N, K, beta != 0.f, lda, ldb, ldc, false);
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
    const int psteps = plane_steps(K);
    int *inexact = nullptr;
    if (p.split >= 2) {
        const int units = plane_cols(N) * psteps;               // (P_MAX_BYTES keeps it small)
        inexact = (int *)(planes + (size_t)units * P_UNIT);
        if (tb) hipLaunchKernelGGL(split_planes_kernel<true>, dim3(units), dim3(64), 0, g_ctx.stream, planes, inexact, B, ldb, N, K, psteps);
        else hipLaunchKernelGGL(split_planes_kernel<false>, dim3(units), dim3(64), 0, g_ctx.stream, planes, inexact, B, ldb, N, K, psteps);
        LAUNCH_OK("sgemm planes");
    }
    auto launch_planes = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)tiles * p.slices), dim3(P_THREADS), 0, g_ctx.stream, A, lda, B, ldb, C, ldc, M, N,
                           k_all, p.k_slice, tiles_n, tiles, alpha, beta, part, (const char *)planes, (const int *)inexact, psteps);
    };
#define GEMM_CASE(BM, BN, WM, WN, KS)                                                                                 \
    case gemm_key(0, KS, BM, BN): {                                                                                   \
        constexpr int threads = GemmShape<BM, BN, WM, WN, KS>::THREADS;                                               \
        if (!ta && !tb) launch(sgemm_kernel<BM, BN, WM, WN, KS, false, false>, threads);                              \
        else if (!ta) launch(sgemm_kernel<BM, BN, WM, WN, KS, false, true>, threads);                                 \
        else if (!tb) launch(sgemm_kernel<BM, BN, WM, WN, KS, true, false>, threads);                                 \
        else launch(sgemm_kernel<BM, BN, WM, WN, KS, true, true>, threads);                                           \
        break;                                                                                                        \
    }
#define SMALL_CASE(BM, BN, WM, WN, KS)                                                                                \
    case gemm_key(1, KS, BM, BN):                                                                                     \
        if (!ta && !tb) launch(sgemm_split_small_kernel<BM, BN, WM, WN, KS, false, false>, SS_THREADS * KS);          \
        else if (!ta) launch(sgemm_split_small_kernel<BM, BN, WM, WN, KS, false, true>, SS_THREADS * KS);             \
        else if (!tb) launch(sgemm_split_small_kernel<BM, BN, WM, WN, KS, true, false>, SS_THREADS * KS);             \
        else launch(sgemm_split_small_kernel<BM, BN, WM, WN, KS, true, true>, SS_THREADS * KS);                       \
        break;
#define SPLIT_CASE(BM, BN)                                                                                            \
    case gemm_key(1, 1, BM, BN):                                                                                      \
        if (!ta && !tb) launch(sgemm_split_kernel<BM, BN, false, false>, S_THREADS);                              \
        else if (!ta) launch(sgemm_split_kernel<BM, BN, false, true>, S_THREADS);                                 \
        else if (!tb) launch(sgemm_split_kernel<BM, BN, true, false>, S_THREADS);                                 \
        else launch(sgemm_split_kernel<BM, BN, true, true>, S_THREADS);                                           \
        break;
    auto launch_rows = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(ceil_div((size_t)M, (size_t)p.bm) * p.ranges)), dim3(R_THREADS), 0, g_ctx.stream, A, lda,
                           B, ldb, C, ldc, M, N, K, p.bn / 32, p.ranges, alpha, beta, (const char *)planes,
                           (const int *)inexact, psteps);
    };
#define ROWS_CASE(FM)                                                                                                 \
    if (p.split == 3 && p.bm == 16 * FM) {                                                                            \
        if (!ta && !tb) launch_rows(sgemm_rows_kernel<FM, false, false>);                                             \
        else if (!ta) launch_rows(sgemm_rows_kernel<FM, false, true>);                                                \
        else if (!tb) launch_rows(sgemm_rows_kernel<FM, true, false>);                                                \
        else launch_rows(sgemm_rows_kernel<FM, true, true>);                                                          \
    } else
#define PLANES_CASE(BM)                                                                                               \
    case gemm_key(2, 1, BM, PN):                                                                                      \
        if (!ta && !tb) launch_planes(sgemm_planes_kernel<BM, false, false>);                                         \
        else if (!ta) launch_planes(sgemm_planes_kernel<BM, false, true>);                                            \
        else if (!tb) launch_planes(sgemm_planes_kernel<BM, true, false>);                                            \
        else launch_planes(sgemm_planes_kernel<BM, true, true>);                                                      \
        break;
    ROWS_CASE(6)
    ROWS_CASE(4)
    switch (gemm_key(p.split, p.groups, p.bm, p.bn)) {
        GEMM_CASE(64, 64, 32, 32, 1)
        GEMM_CASE(64, 64, 32, 32, 2)
        GEMM_CASE(64, 32, 32, 32, 4)
        GEMM_CASE(32, 64, 32, 32, 4)
        SMALL_CASE(64, 64, 32, 32, 1)
        SMALL_CASE(64, 64, 32, 32, 2)
        SPLIT_CASE(128, 256)
        SPLIT_CASE(256, 128)
        PLANES_CASE(96)
        PLANES_CASE(64)
        default: return mi355_fail("sgemm: no kernel for a tile of %d x %d", p.bm, p.bn);
    }
#undef GEMM_CASE
#undef SMALL_CASE
#undef SPLIT_CASE
#undef PLANES_CASE
#undef ROWS_CASE
    LAUNCH_OK("sgemm");
    if (part) {
        auto sum = [&](auto kernel, int groups) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div((size_t)M * N, 256 / groups)), dim3(256), 0, g_ctx.stream, C, ldc,
                               part, p.slices, M, N, alpha, beta);
        };
        if (p.slices <= 8 || (size_t)M * N > 65536) sum(slice_sum_kernel<1>, 1);
        else sum(slice_sum_kernel<16>, 16);
        LAUNCH_OK("sgemm slice sum");
    }
    return 0;
}

}   // namespace

void mi355_free_planes(void) {
    if (!g_planes) return;
    (void)hipStreamSynchronize(g_ctx.stream);
    (void)hipFree(g_planes);
    g_planes = nullptr;
    g_planes_bytes = 0;
}

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
    // columns as make 2^21 tiles of 64 x 64 (of 512 threads, and twice as many where a tile is half as large).  All but thin
    // products of many millions of rows or columns, long ones of a billion k and outputs beyond 32 GB are one piece.
    constexpr int KC = 1 << 30, MC = 1 << 26;
    const int mc = M < MC ? M : MC;
    const size_t tiles_n = ((size_t)1 << 21) / ceil_div((size_t)mc, 64);
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
