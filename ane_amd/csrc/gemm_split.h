// gemm_split.h — fp32 products on the bfloat16 matrix instruction.  Included by gemm.hip inside its unnamed namespace.
//
// An fp32 value is the sum of three bfloat16 values, exactly: h = the value rounded to 8 bits, m = what is left rounded
// to 8 bits, l = the rest (24 bits in three signed groups of 8).  Of the nine products of two such sums the six down to
// 2^-16 of the first are taken (hh, hm, mh, hl, lh, mm), each with an exact fp32 product and fp32 sums in
// v_mfma_f32_16x16x32_bf16; what is left out is below 2^-24 of a term.  Six instructions of 32 terms stand for eight of
// v_mfma_f32_16x16x4_f32, take 6 x 16 cycles instead of 8 x 32, and round a sum six times where those round it eight
// times.  Against 64 bits the error of the large tiles is smaller from K = 80 on, that of the small ones, which keep a sum of
// their own for the hh products, a third at any K (figures at plan_gemm).
// A split is not exact where l leaves bfloat16 (values below 2^-109), and h + m + l of an infinity or of a value that
// rounds to one is a NaN.  Both are seen: the first in the low half of l's pattern, the second in the result, which is
// then not finite.  A workgroup that saw either computes its tile again with the fp32 instruction, straight from memory
// (about twice the time), so such values give what they give there.
//
// A workgroup of eight waves owns a tile of 128 x 256 or 256 x 128, a wave 64 x 64 of it, and K goes in steps of 32 through
// two LDS buffers of three planes each (147 KB).  A row of a plane is 32 values of k in 64 bytes, for both operands and all
// transpose cases: a thread has eight values of k of a row in registers when it splits them (K contiguous: two 128-bit
// loads; K strided: one load of W columns from each of eight rows), and 16 bytes per plane are what it writes and what a
// lane of the instruction reads.  Rows lie in LDS as split_slot says, so that the four fragments of a wave give a lane
// four neighbouring columns of C; the 16-byte chunks of a row are permuted (split_chunk) against bank conflicts.
// A step takes 2.45 us where its instructions take 1.28 at 2.4 GHz; the chip runs this kernel at 1.8 GHz, so the matrix
// cores are busy 70 % of the time.  The splitting (6 vector instructions per value) is a third of the matrix time and runs
// in the shadow of the other wave of the SIMD; with the whole splitting at the end of a step and the barrier behind it,
// 4096 x 4096 x 4096 took 667 us, in this order 640 (215 TFLOP/s; the fp32 instruction 1145 us).
#pragma once

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));

constexpr int SK = 32;                 // K per step
constexpr int S_THREADS = 512;

// Chunk c of the row at `slot`.  A 128-bit LDS read goes in groups of sixteen lanes, 0-3, 12-15, 20-23 and 24-27 the first:
// rows 0-3 and 12-15 of one chunk with rows 4-11 of the next; writes go sixteen lanes in order.
__device__ __forceinline__ int split_chunk(int slot, int c) {
    const int a = slot >> 2, g = ((a >> 1) & 1) | (((a ^ (a >> 1)) & 1) << 1);
    return c ^ g ^ ((slot >> 4) & 3);
}
// F fragments (16 rows each) to a wave: row F*i + j of a group of 16*F lies at 16j + i
template <int F>
__device__ __forceinline__ int split_slot(int x) { return (x & ~(16 * F - 1)) | (x & (F - 1)) << 4 | ((x / F) & 15); }
template <int F>
__device__ __forceinline__ int split_row(int slot) { return (slot & ~(16 * F - 1)) | (slot & 15) * F | ((slot >> 4) & (F - 1)); }

struct Planes { v4u h, m, l; };
// splits values 2 j0 .. 2 j1 - 1 of a piece; the low half of `left` takes what a split could not hold
__device__ __forceinline__ void split_eight(const float (&r)[8], int j0, int j1, Planes &o, unsigned &left) {
#pragma unroll
    for (int j = j0; j < j1; j++) {
        float a = r[2 * j], b = r[2 * j + 1];
        o.h[j] = f2_to_bf2(a, b);
        a -= bf_to_f(o.h[j]);
        b -= __uint_as_float(o.h[j] & 0xffff0000u);
        o.m[j] = f2_to_bf2(a, b);
        a -= bf_to_f(o.m[j]);
        b -= __uint_as_float(o.m[j] & 0xffff0000u);
        o.l[j] = f2_to_bf2(a, b);
        left |= __float_as_uint(a) | __float_as_uint(b);
    }
}

// One operand tile of BX rows (of M or N) by SK: global -> registers -> three planes in LDS.  KC: k is the contiguous index.
// THREADS: of the group of waves that loads it, tid() a thread's number in the group; groups take the steps in turn.
template <int BX, bool KC, int THREADS, int F>
struct SplitOperand {
    static constexpr int PIECES = BX * (SK / 8);                             // eight values of k of one row
    static constexpr int NP = PIECES / THREADS;                              // per thread
    static constexpr int W = NP;                                             // K strided: columns of one load
    static constexpr int PLANE = BX * SK * 2;                                // bytes
    static_assert(PIECES % THREADS == 0 && (W == 1 || W == 2), "whole pieces, units of W columns");
    const char *base;           // the step at hand (the same for the whole workgroup)
    size_t ahead;               // bytes from one step to the next
    size_t row;                 // K strided: bytes from one k to the next
    unsigned off[NP];           // this thread's pieces (K strided: the columns of its unit)
    int kc;                     // first k of the thread's pieces / 8
    float r[NP][8];

    // K contiguous: four threads to a row.  K strided: sixteen threads cover 16 columns and W chunks of k.
    static __device__ __forceinline__ int tid() { return threadIdx.x % THREADS; }
    static __device__ __forceinline__ int unit_x() {
        const int g = tid() >> 4;
        return g % (BX / 16) * 16 + (tid() & 15) % (16 / W) * W;
    }
    static __device__ __forceinline__ int piece_slot(int p) {
        return KC ? (tid() >> 2) + p * (THREADS / 4) : split_slot<F>(unit_x() + p);
    }

    // rows past the end are read from the last one; what they multiply is never stored
    __device__ __forceinline__ void start(const float *__restrict__ p, int ld, int x0, int X, int k0, int groups = 1) {
        if constexpr (KC) {
            kc = tid() & 3;
#pragma unroll
            for (int i = 0; i < NP; i++) {
                const int x = min(x0 + split_row<F>(piece_slot(i)), X - 1) - x0;
                off[i] = ((unsigned)x * (unsigned)ld + 8 * kc) * 4;
            }
            base = (const char *)(p + (size_t)x0 * ld + k0);
            ahead = (size_t)SK * 4 * groups;
            row = 4;
        } else {
            kc = (tid() >> 4) / (BX / 16) * W + (tid() & 15) / (16 / W);
#pragma unroll
            for (int i = 0; i < NP; i++)
                off[i] = ((unsigned)(8 * kc) * (unsigned)ld + (unsigned)(min(x0 + unit_x() + i, X - 1) - x0)) * 4;
            base = (const char *)(p + (size_t)k0 * ld + x0);
            ahead = (size_t)SK * ld * 4 * groups;
            row = (size_t)ld * 4;
        }
    }
    // the pieces of a whole step; edge: the tile hangs over the end of the rows (the same for the whole workgroup)
    __device__ __forceinline__ void fetch(bool edge) {
        if constexpr (KC) {
#pragma unroll
            for (int i = 0; i < NP; i++)
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const v4f v = ld4((const float *)(base + off[i]) + 4 * q);
#pragma unroll
                    for (int j = 0; j < 4; j++) r[i][4 * q + j] = v[j];
                }
        } else if (W == 1 || edge) {
#pragma unroll
            for (int k = 0; k < 8; k++)
#pragma unroll
                for (int i = 0; i < NP; i++) r[i][k] = *(const float *)(base + k * row + off[i]);
        } else {
            typedef float v2f_any __attribute__((ext_vector_type(2), aligned(4)));
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const v2f v = *(const v2f_any *)(base + k * row + off[0]);
                r[0][k] = v[0];
                r[NP - 1][k] = v[1];
            }
        }
        base += ahead;
    }
    // the pieces of a step of which only n < SK values of k exist
    __device__ __forceinline__ void fetch_tail(int n) {
#pragma unroll
        for (int i = 0; i < NP; i++)
#pragma unroll
            for (int k = 0; k < 8; k++) r[i][k] = 8 * kc + k < n ? *(const float *)(base + k * row + off[i]) : 0.f;
    }
    __device__ __forceinline__ void split(int p, int j0, int j1, Planes &o, unsigned &left) const {
        split_eight(r[p], j0, j1, o, left);
    }
    __device__ __forceinline__ void write(int p, const Planes &o, char *lds) const {
        const int slot = piece_slot(p);
        char *to = lds + slot * (SK * 2) + split_chunk(slot, kc) * 16;
        *reinterpret_cast<v4u *>(to) = o.h;
        *reinterpret_cast<v4u *>(to + PLANE) = o.m;
        *reinterpret_cast<v4u *>(to + 2 * PLANE) = o.l;
    }
};

// The wave's fragments at rows m0.. and columns n0.., over k_beg .. k_end, again with the fp32 instruction.
// Register e of a lane's fragment i, j: row FM * (4 * quarter + e) + i, column FN * li + j; ROWS16: row 16 * i + 4 * quarter + e.
template <int FM, int FN, bool TA, bool TB, bool ROWS16>
__device__ __forceinline__ void split_again(v4f (&acc)[FM][FN], const float *__restrict__ A, int lda,
                                            const float *__restrict__ B, int ldb, int M, int N, int m0, int n0, int k_beg,
                                            int k_end) {
    const int lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;
    const float *pa[FM], *pb[FN];
#pragma unroll
    for (int i = 0; i < FM; i++) {
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        const int m = min(m0 + (ROWS16 ? 16 * i + li : FM * li + i), M - 1);
        pa[i] = TA ? A + m : A + (size_t)m * lda;
    }
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const int nn = min(n0 + FN * li + j, N - 1);
        pb[j] = TB ? B + (size_t)nn * ldb : B + nn;
    }
    for (int k0 = k_beg; k0 < k_end; k0 += 4) {
        const int k = k0 + quarter;
        float va[FM], vb[FN];
#pragma unroll
        for (int i = 0; i < FM; i++) va[i] = k < k_end ? pa[i][TA ? (size_t)k * lda : (size_t)k] : 0.f;
#pragma unroll
        for (int j = 0; j < FN; j++) vb[j] = k < k_end ? pb[j][TB ? (size_t)k : (size_t)k * ldb] : 0.f;
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[i], vb[j], acc[i][j], 0, 0, 0);
    }
}
template <int FM, int FN>
__device__ __forceinline__ bool split_not_finite(const v4f (&acc)[FM][FN]) {
    bool again = false;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) again |= (__float_as_uint(acc[i][j][e]) & 0x7f800000u) == 0x7f800000u;
    return again;
}

// The end of a tile: the wave's fragments at rows m0.. and columns n0.., computed again where values called for it
// (`left`: what the splits could not hold), scaled and stored; part: where the bare product of the slice goes, or NULL;
// mine: this wave finishes them.
template <int FM, int FN, bool TA, bool TB, bool ROWS16 = false>
__device__ __forceinline__ void split_finish(v4f (&acc)[FM][FN], unsigned left, const float *__restrict__ A, int lda,
                                             const float *__restrict__ B, int ldb, float *C, int ldc, int M, int N, int m0,
                                             int n0, int k_beg, int k_end, float alpha, float beta, float *__restrict__ part,
                                             bool mine = true) {
    typedef float vec __attribute__((ext_vector_type(FN), aligned(4)));
    const int lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;
    const int n = n0 + FN * li;
    const bool bad = __syncthreads_or((left & 0xffffu) != 0 || split_not_finite<FM, FN>(acc));
    if (!mine) return;
    if (bad) split_again<FM, FN, TA, TB, ROWS16>(acc, A, lda, B, ldb, M, N, m0, n0, k_beg, k_end);

    float *out = part ? part : C;
    const int ldo = part ? N : ldc;
    const bool read = !part && beta != 0.f;             // beta == 0 does not read C (cblas semantics)
    vec c[FM][4];                                       // all of the old values are asked for before the first store
    auto each = [&](auto fn) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int m = m0 + (ROWS16 ? 16 * i + 4 * quarter + e : FM * (4 * quarter + e) + i);
                if (m < M) fn(i, e, out + (size_t)m * ldo + n);
            }
    };
    if (read)
        each([&](int i, int e, const float *o) {
            if (n + FN <= N) {
                c[i][e] = *reinterpret_cast<const vec *>(o);
            } else {
#pragma unroll
                for (int j = 0; j < FN; j++) c[i][e][j] = n + j < N ? o[j] : 0.f;
            }
        });
    each([&](int i, int e, float *o) {
        vec v;
#pragma unroll
        for (int j = 0; j < FN; j++) v[j] = part ? acc[i][j][e] : acc[i][j][e] * alpha;
        if (read) v += beta * c[i][e];
        if (n + FN <= N) {
            *reinterpret_cast<vec *>(o) = v;
        } else {
#pragma unroll
            for (int j = 0; j < FN; j++)
                if (n + j < N) o[j] = v[j];
        }
    });
}

// C = alpha * op(A) . op(B) + beta * C for one K slice; part != NULL: the bare product of the slice goes to part[slice].
// Workgroup order as sgemm_kernel's.  lda, ldb < 2^22: the lanes' offsets into a tile are 32 bits of bytes.
template <int BM, int BN, bool TA, bool TB>
__global__ __launch_bounds__(S_THREADS) void sgemm_split_kernel(const float *__restrict__ A, int lda,
                                                                const float *__restrict__ B, int ldb, float *C, int ldc,
                                                                int M, int N, int K, int k_slice, int tiles_n, int tiles,
                                                                float alpha, float beta, float *__restrict__ part) {
    constexpr int WM = 64, WN = 64, FM = WM / 16, FN = WN / 16;
    typedef SplitOperand<BM, !TA, S_THREADS, FM> OpA;
    typedef SplitOperand<BN, TB, S_THREADS, FN> OpB;
    static_assert((BM / WM) * (BN / WN) == S_THREADS / 64, "eight waves cover the tile");
    __shared__ __align__(16) char lds[2][3 * (OpA::PLANE + OpB::PLANE)];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int slice = logical / tiles, tile = logical - slice * tiles;
    const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * BN;
    const int k_beg = slice * k_slice, k_end = min(K, k_beg + k_slice);
    const int steps = (k_end - k_beg) / SK, rest = (k_end - k_beg) % SK, all = steps + (rest > 0);
    const bool edge_m = m0 + BM > M, edge_n = n0 + BN > N;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;
    const int wm = wave / (BN / WN) * WM, wn = wave % (BN / WN) * WN;

    v4f acc[FM][FN];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    unsigned left = 0;
    OpA oa;
    OpB ob;
    oa.start(A, lda, m0, M, k_beg);
    ob.start(B, ldb, n0, N, k_beg);
    auto fetch = [&](int t) {
        if (t < steps) { oa.fetch(edge_m); ob.fetch(edge_n); }
        else { oa.fetch_tail(rest); ob.fetch_tail(rest); }
    };
    constexpr int NPA = OpA::NP, NPB = OpB::NP;
    static_assert(NPA + NPB < FN, "a step's pieces go between the columns of products, before the last");
    auto split = [&](int p, int j0, int j1, Planes &o) {
        if (p < NPA) oa.split(p < NPA ? p : 0, j0, j1, o, left);
        else ob.split(p < NPA ? 0 : p - NPA, j0, j1, o, left);
    };
    auto write = [&](int p, const Planes &o, char *to) {
        if (p < NPA) oa.write(p < NPA ? p : 0, o, to);
        else ob.write(p < NPA ? 0 : p - NPA, o, to + 3 * OpA::PLANE);
    };
    int fa[FM], fb[FN];                                  // where this lane's fragments lie in a plane
#pragma unroll
    for (int i = 0; i < FM; i++) {
        const int slot = wm + 16 * i + li;
        fa[i] = slot * (SK * 2) + split_chunk(slot, quarter) * 16;
    }
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const int slot = wn + 16 * j + li;
        fb[j] = slot * (SK * 2) + split_chunk(slot, quarter) * 16 + 3 * OpA::PLANE;
    }
    fetch(0);
#pragma unroll
    for (int p = 0; p < NPA + NPB; p++) {
        Planes o;
        split(p, 0, 4, o);
        write(p, o, lds[0]);
    }
    if (all > 1) fetch(1);
    __syncthreads();
    bf8_t a[FM][3], b[FN][3];
    auto read_a = [&](const char *buf, int q) {
#pragma unroll
        for (int i = 0; i < FM; i++) a[i][q] = *reinterpret_cast<const bf8_t *>(buf + fa[i] + q * OpA::PLANE);
    };
    auto read_b = [&](const char *buf, int j, int q) { b[j][q] = *reinterpret_cast<const bf8_t *>(buf + fb[j] + q * OpB::PLANE); };
    auto products = [&](int j, int p0, int p1) {
        constexpr int P[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 0}, {1, 1}, {2, 0}};
#pragma unroll
        for (int p = p0; p < p1; p++)
#pragma unroll
            for (int i = 0; i < FM; i++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][P[p][0]], b[j][P[p][1]], acc[i][j], 0, 0, 0);
    };
    auto read_first = [&](const char *buf) { read_a(buf, 0); read_b(buf, 0, 0); read_b(buf, 0, 1); };
    if (all > 0) read_first(lds[0]);
    // A step: the products of the tile in one buffer.  Between them the next tile's values, which are in registers, are
    // split and written to the other buffer, half a piece behind every twelve products: the two waves of a SIMD then split
    // and multiply in turns.  The barrier stands before the last column of products, when all of the tile is in
    // registers; behind it the first fragments of the next tile are read as soon as their registers are free, so the
    // products do not stop for them.
    for (int t = 0; t < all; t++) {
        const char *cur = lds[t & 1];
        char *next = lds[(t + 1) & 1];
        read_b(cur, 0, 2); read_a(cur, 1); read_a(cur, 2);
        auto columns = [&](auto more) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j + 1 < FN; j++) {
                const bool piece = decltype(more)::value && j < NPA + NPB;
                Planes o;
                read_b(cur, j + 1, 0); read_b(cur, j + 1, 1); read_b(cur, j + 1, 2);
                products(j, 0, 3);
                __builtin_amdgcn_sched_barrier(0);
                if (piece) split(j, 0, 2, o);
                __builtin_amdgcn_sched_barrier(0);
                products(j, 3, 6);
                __builtin_amdgcn_sched_barrier(0);
                if (piece) {
                    split(j, 2, 4, o);
                    write(j, o, next);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (t + 1 < all) {
            columns(std::true_type());
            __syncthreads();
            products(FN - 1, 0, 3);
            __builtin_amdgcn_sched_barrier(0);
            read_first(next);
            __builtin_amdgcn_sched_barrier(0);
            products(FN - 1, 3, 6);
            __builtin_amdgcn_sched_barrier(0);
            if (t + 2 < all) fetch(t + 2);
        } else {
            columns(std::false_type());
            products(FN - 1, 0, 6);
        }
    }

    split_finish<FM, FN, TA, TB>(acc, left, A, lda, B, ldb, C, ldc, M, N, m0 + wm, n0 + wn, k_beg, k_end, alpha, beta,
                                 part ? part + (size_t)slice * M * N : nullptr);
}

// The same for outputs with few tiles of 128 x 256: KS groups of four waves own a tile of 64 x 64 (a wave 32 x 32) and take the
// steps in turn.  One group: three workgroups share a compute unit (49 KB each) and one splits, loads or stores while another
// multiplies; [3072][256] . [256][1024] += 18.0 us (fp32 64 x 64 20.1, 128 x 256 27), [9001][768] . [768][197] 35 (49, 43).
// Two groups: where there is one tile to a compute unit, whose four waves would wait for each other (1024 x 1024 x 1024
// 27.8 with one group, 21.6 with two).  There the steps up to the last few know that there is another behind them: a step
// without branches can be scheduled as one ([3563][1024] . [1024][256] 22.0 -> 20.1 us, [2657][768] . [768][256] 16.7 -> 14.9); with one
// group, where other workgroups fill in, that changes nothing or costs
// ([9001][1024] . [1024][256] 44 -> 50).  What bounds it is the splitting, done again by every tile: at 64 x 64 as many vector
// cycles as half of the matrix cycles, and the LDS reads, as many cycles as the products.  A second step on its way to
// registers changed nothing (12.7 and 12.7 at [2048][256] . [256][768]), nor did tiles of 64 x 128 (13.4).
// The hh products of a term have sums of their own, so a sum of full size is rounded once per 32 values of k, and the five
// small products, below 2^-8 of it, beside it.
constexpr int SS_THREADS = 256;        // of a group
template <int BM, int BN, int WM, int WN, int KS, bool TA, bool TB>
__global__ __launch_bounds__(SS_THREADS * KS) void sgemm_split_small_kernel(const float *__restrict__ A, int lda,
                                                                            const float *__restrict__ B, int ldb, float *C,
                                                                            int ldc, int M, int N, int K, int k_slice,
                                                                            int tiles_n, int tiles, float alpha, float beta,
                                                                            float *__restrict__ part) {
    constexpr int FM = WM / 16, FN = WN / 16;
    typedef SplitOperand<BM, !TA, SS_THREADS, FM> OpA;
    typedef SplitOperand<BN, TB, SS_THREADS, FN> OpB;
    static_assert((BM / WM) * (BN / WN) == SS_THREADS / 64, "four waves cover the tile");
    __shared__ __align__(16) char lds[KS][2][3 * (OpA::PLANE + OpB::PLANE)];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int slice = logical / tiles, tile = logical - slice * tiles;
    const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * BN;
    const int k_beg = slice * k_slice, k_end = min(K, k_beg + k_slice);
    const int steps = (k_end - k_beg) / SK, rest = (k_end - k_beg) % SK, all = steps + (rest > 0);
    const bool edge_m = m0 + BM > M, edge_n = n0 + BN > N;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;
    const int group = wave / 4, ww = wave % 4;
    const int wm = ww / (BN / WN) * WM, wn = ww % (BN / WN) * WN;

    v4f acc[FM][FN], low[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = low[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    unsigned left = 0;
    OpA oa;
    OpB ob;
    oa.start(A, lda, m0, M, k_beg + SK * group, KS);
    ob.start(B, ldb, n0, N, k_beg + SK * group, KS);
    // step t of the group is step KS * t + group of the tile; where that is past the end it is all zeros
    const int rounds = (all + KS - 1) / KS;
    auto fetch = [&](int t) {
        const int s = KS * t + group;
        if (s < steps) { oa.fetch(edge_m); ob.fetch(edge_n); }
        else { oa.fetch_tail(s == steps ? rest : 0); ob.fetch_tail(s == steps ? rest : 0); }
    };
    constexpr int NPA = OpA::NP, NPB = OpB::NP;
    auto piece = [&](int p, char *to) {
        Planes o;
        if (p < NPA) {
            oa.split(p < NPA ? p : 0, 0, 4, o, left);
            oa.write(p < NPA ? p : 0, o, to);
        } else {
            ob.split(p < NPA ? 0 : p - NPA, 0, 4, o, left);
            ob.write(p < NPA ? 0 : p - NPA, o, to + 3 * OpA::PLANE);
        }
    };
    fetch(0);
#pragma unroll
    for (int p = 0; p < NPA + NPB; p++) piece(p, lds[group][0]);
    if (rounds > 1) fetch(1);
    __syncthreads();
    int fa[FM], fb[FN];                                  // where this lane's fragments lie in a plane
#pragma unroll
    for (int i = 0; i < FM; i++) {
        const int slot = wm + 16 * i + li;
        fa[i] = slot * (SK * 2) + split_chunk(slot, quarter) * 16;
    }
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const int slot = wn + 16 * j + li;
        fb[j] = slot * (SK * 2) + split_chunk(slot, quarter) * 16 + 3 * OpA::PLANE;
    }
    auto step = [&](auto steady, int t) __attribute__((always_inline)) {
        const char *cur = lds[group][t & 1];
        bf8_t a[FM][3], b[FN][3];
#pragma unroll
        for (int q = 0; q < 3; q++) {
#pragma unroll
            for (int i = 0; i < FM; i++) a[i][q] = *reinterpret_cast<const bf8_t *>(cur + fa[i] + q * OpA::PLANE);
#pragma unroll
            for (int j = 0; j < FN; j++) b[j][q] = *reinterpret_cast<const bf8_t *>(cur + fb[j] + q * OpB::PLANE);
        }
        const bool more = decltype(steady)::value || t + 1 < rounds;
        constexpr int P[6][2] = {{0, 0}, {0, 1}, {1, 0}, {1, 1}, {0, 2}, {2, 0}};
#pragma unroll
        for (int p = 0; p < 6; p++) {
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) {
                    v4f &s = p == 0 ? acc[i][j] : low[i][j];
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][P[p][0]], b[j][P[p][1]], s, 0, 0, 0);
                }
            if (more && p < NPA + NPB) piece(p, lds[group][(t + 1) & 1]);
        }
        if (decltype(steady)::value) { oa.fetch(edge_m); ob.fetch(edge_n); }
        else if (t + 2 < rounds) fetch(t + 2);
        if (more) __syncthreads();
    };
    int t = 0;
    if constexpr (KS > 1)
        for (; KS * (t + 2) + KS - 1 < steps; t++) step(std::true_type(), t);
    for (; t < rounds; t++) step(std::false_type(), t);
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] += low[i][j];
    if constexpr (KS > 1) {
        // the other groups' sums, added in group order by the first; they leave with it at the next barrier
        static_assert((KS - 1) * BM * BN * 4 <= (int)sizeof(lds), "the sums fit the buffers");
        v4f *x = reinterpret_cast<v4f *>(&lds[0][0][0]);
        auto at = [&](int g, int f) { return ((g - 1) * FM * FN + f) * SS_THREADS + ww * 64 + lane; };
        __syncthreads();
        if (group > 0) {
#pragma unroll
            for (int f = 0; f < FM * FN; f++) x[at(group, f)] = acc[f / FN][f % FN];
        }
        __syncthreads();
        if (group == 0) {
#pragma unroll
            for (int g = 1; g < KS; g++)
#pragma unroll
                for (int f = 0; f < FM * FN; f++) acc[f / FN][f % FN] += x[at(g, f)];
        }
    }
    split_finish<FM, FN, TA, TB>(acc, left, A, lda, B, ldb, C, ldc, M, N, m0 + wm, n0 + wn, k_beg, k_end, alpha, beta,
                                 part ? part + (size_t)slice * M * N : nullptr, group == 0);
}
