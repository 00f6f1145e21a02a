// gemm_planes.h — fp32 products on the bfloat16 matrix instruction, the smaller operand split ahead of the product.
// Included by gemm.hip inside its unnamed namespace, behind gemm_split.h (whose comment says what a split is).
//
// The tiles of gemm_split.h split both operands of a tile again in every tile.  In the classifier's products one operand
// is small and every tile needs it ([24573][1024] . [1024][256]: 192 tiles, each of which splits all of the 1024 x 256),
// two thirds of the splitting and of the LDS writes.  Here a launch of its own (split_planes_kernel, 4 us for 1 MB) splits B
// once, into three planes that lie in memory as the fragments of the instruction: a wave of the product loads a fragment with one
// contiguous 1 KB access straight into the registers of the instruction, through neither LDS nor vector instructions, and no two
// waves of a workgroup load the same one.
// Both kernels have sixteen waves of 16 * FM x 32 of the output, four on a SIMD with 128 registers each, so that one
// waits for B, old values of C or its stores while others multiply.  With eight waves, B asked for a step ahead and 256 registers
// each, [24573][1024] . [1024][256] took 70 us, [24573][256] . [256][1024] += 77 (16 waves: 65 and 67).
// What bounds them: with everything but the products left out these two take 55 and 53 us of 70 and 68 (33 for the
// instructions alone at 2.35 PFLOP/s, the rest the launches, the first loads and the last stores).
#pragma once

constexpr int PK = 64;                 // K per step
constexpr int PN = 256;                // columns of a tile
constexpr int P_THREADS = 1024;
constexpr int P_FRAG = 1024;           // bytes of a fragment of a plane: 64 lanes x 8 values
constexpr int P_UNIT = 6 * P_FRAG;     // 32 columns by 32 values of k: two fragments of three planes
constexpr size_t P_MAX_BYTES = (size_t)256 << 20;       // the planes of a call; larger operands take the other kernels

// Units of the planes of a K x N operand: [unit of 32 columns][step of 32 k][fragment][plane][lane]; columns and k are filled
// up with zeros to whole tiles and steps.
static inline int plane_cols(int N) { return (int)ceil_div((size_t)N, PN) * (PN / 32); }
static inline int plane_steps(int K) { return (int)ceil_div((size_t)K, PK) * 2; }
static inline size_t plane_bytes(int N, int K) { return (size_t)plane_cols(N) * plane_steps(K) * (P_UNIT + sizeof(int)); }

// B -> planes; inexact[unit]: whether a value of the unit is not the sum of its three parts.  A wave takes a unit: fragment j of
// lane l holds column 2 * (l % 16) + j and the eight values of k from 8 * (l / 16) on.
// A wave to a workgroup, so that an operand of 1 MB has one for every compute unit, and nothing of a unit that lies inside B behind a
// condition (four to a workgroup, every load behind its row of k: [1024][256] ahead of a product of 24573 rows 2 us longer in all).
template <bool TB>
__global__ __launch_bounds__(64) void split_planes_kernel(char *__restrict__ planes, int *__restrict__ inexact,
                                                           const float *__restrict__ B, int ldb, int N, int K, int steps) {
    const int unit = blockIdx.x, lane = threadIdx.x, cu = unit / steps, s = unit - cu * steps;
    const bool inside = cu * 32 + 32 <= N && s * 32 + 32 <= K;
    const int n = cu * 32 + 2 * (lane & 15), k = s * 32 + 8 * (lane >> 4);
    typedef float v2f_any __attribute__((ext_vector_type(2), aligned(4)));
    float r[2][8];
    if (inside) {
        const float *p = B + (TB ? (size_t)n * ldb + k : (size_t)k * ldb + n);
        if constexpr (TB) {
            v4f a[2][2];
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int h = 0; h < 2; h++) a[j][h] = ld4(p + (size_t)j * ldb + 4 * h);
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 8; e++) r[j][e] = a[j][e / 4][e & 3];
        } else {
            v2f a[8];
#pragma unroll
            for (int e = 0; e < 8; e++) a[e] = *(const v2f_any *)(p + (size_t)e * ldb);
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 8; e++) r[j][e] = a[e][j];
        }
    } else if constexpr (TB) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float *p = B + (size_t)min(n + j, N - 1) * ldb + k;
            if (k + 8 <= K) {
                const v4f a = ld4(p), b = ld4(p + 4);
#pragma unroll
                for (int e = 0; e < 4; e++) { r[j][e] = a[e]; r[j][4 + e] = b[e]; }
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) r[j][e] = k + e < K ? p[e] : 0.f;
            }
            if (n + j >= N) {
#pragma unroll
                for (int e = 0; e < 8; e++) r[j][e] = 0.f;
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            r[0][e] = r[1][e] = 0.f;
            if (k + e < K) {
                const float *p = B + (size_t)(k + e) * ldb + n;
                if (n + 1 < N) {
                    const v2f v = *(const v2f_any *)p;
                    r[0][e] = v[0];
                    r[1][e] = v[1];
                } else if (n < N) {
                    r[0][e] = p[0];
                }
            }
        }
    }
    unsigned left = 0;
    char *to = planes + (size_t)unit * P_UNIT + lane * 16;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        Planes o;
        split_eight(r[j], 0, 4, o, left);
        *reinterpret_cast<v4u *>(to + (3 * j + 0) * P_FRAG) = o.h;
        *reinterpret_cast<v4u *>(to + (3 * j + 1) * P_FRAG) = o.m;
        *reinterpret_cast<v4u *>(to + (3 * j + 2) * P_FRAG) = o.l;
    }
    const bool any = __builtin_amdgcn_ballot_w64((left & 0xffffu) != 0) != 0;
    if (lane == 0) inexact[unit] = any;
}

// The tile of A: BM rows by PK values of k, global -> registers -> three planes in LDS, fragment by fragment:
// [32 k][16 rows][plane][64 x 16 bytes].  Slot (quarter q of k, row r of 16) lies at 16q + (r ^ 2 * (4 * (k / 32) + q)): an
// eight-lane row of a write (KC: all of a row's k) then goes to eight different banks, two rows to sixteen, and the sixteen lanes
// that a read serves at a time (see split_chunk) still find sixteen.
// A thread has one piece of eight values of k; where there are fewer pieces than threads, the last waves have none.
template <int BM, bool KC>
struct PlaneOperand {
    static constexpr int PIECES = BM * (PK / 8);
    static constexpr int FM = BM / 16;
    static constexpr int BYTES = 2 * FM * 3 * P_FRAG;
    static_assert(PIECES <= P_THREADS && PIECES % 64 == 0, "one piece per thread, whole waves");
    const char *base;
    size_t ahead, row;          // bytes from one step to the next, from one k to the next
    unsigned off;
    float r[8];

    static __device__ __forceinline__ void place(int &x, int &c) {      // row of the tile, chunk of eight k
        const int p = min((int)threadIdx.x, PIECES - 1);
        if constexpr (KC) { x = p / (PK / 8); c = p % (PK / 8); }
        else { x = p % BM; c = p / BM; }
    }
    static __device__ __forceinline__ int slot(int ks, int q, int r) { return (16 * q + (r ^ (2 * (4 * ks + q)))) * 16; }
    // rows past the end are read from the last one; what they multiply is never stored
    __device__ __forceinline__ void start(const float *__restrict__ p, int ld, int x0, int X, int k0) {
        int x, c;
        place(x, c);
        x = min(x0 + x, X - 1) - x0;
        off = KC ? ((unsigned)x * (unsigned)ld + 8 * c) * 4 : ((unsigned)(8 * c) * (unsigned)ld + x) * 4;
        base = (const char *)(KC ? p + (size_t)x0 * ld + k0 : p + (size_t)k0 * ld + x0);
        ahead = (size_t)PK * 4 * (KC ? 1 : ld);
        row = KC ? 4 : (size_t)ld * 4;
    }
    // the piece of the step at hand
    __device__ __forceinline__ void fetch() {
        if constexpr (KC) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const v4f v = ld4((const float *)(base + off) + 4 * q);
#pragma unroll
                for (int j = 0; j < 4; j++) r[4 * q + j] = v[j];
            }
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) r[k] = *(const float *)(base + k * row + off);
        }
    }
    // the same of a step that has n < PK values of k and starts `steps` steps behind the one at hand
    __device__ __forceinline__ void fetch_short(int steps, int n) {
        int x, c;
        place(x, c);
        const char *from = base + (size_t)steps * ahead;
#pragma unroll
        for (int k = 0; k < 8; k++) r[k] = 8 * c + k < n ? *(const float *)(from + k * row + off) : 0.f;
    }
    __device__ __forceinline__ void write(const Planes &o, char *lds) const {
        int x, c;
        place(x, c);
        char *to = lds + ((c >> 2) * FM + (x >> 4)) * (3 * P_FRAG) + slot(c >> 2, c & 3, x & 15);
        *reinterpret_cast<v4u *>(to) = o.h;
        *reinterpret_cast<v4u *>(to + P_FRAG) = o.m;
        *reinterpret_cast<v4u *>(to + 2 * P_FRAG) = o.l;
    }
};

// The six products of a fragment of A with FN of B, 32 values of k.  They have a sum of their own, which is added to the tile's
// behind the last: the tile's sum, the large one, is rounded once per 32 values of k and not six times.
// next_a(q), next_b(q): called when the products are through with the registers of plane q, for what the next fragment needs
// there.  The order depends on where among the fragments of a step this one is, so that a plane of A, and behind the last
// one of B, is mostly needed again several products after its registers are free.
enum class Turn { FIRST, MIDDLE, LAST };
template <Turn TURN, int FN, typename NextA, typename NextB>
__device__ __forceinline__ void plane_products(v4f (&tile)[FN], const bf8_t (&a)[3], const bf8_t (&b)[FN][3], NextA next_a,
                                               NextB next_b) {
    constexpr int ORDER[3][6][2] = {{{1, 1}, {0, 2}, {0, 1}, {2, 0}, {1, 0}, {0, 0}},
                                    {{1, 1}, {1, 0}, {2, 0}, {0, 2}, {0, 1}, {0, 0}},
                                    {{0, 2}, {1, 1}, {0, 1}, {2, 0}, {1, 0}, {0, 0}}};
    v4f sum[FN];
#pragma unroll
    for (int p = 0; p < 6; p++) {
        const auto &order = ORDER[(int)TURN];
#pragma unroll
        for (int j = 0; j < FN; j++)
            sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[order[p][0]], b[j][order[p][1]],
                                                             p == 0 ? v4f{0.f, 0.f, 0.f, 0.f} : sum[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        bool again[2] = {false, false};
#pragma unroll
        for (int q = p + 1; q < 6; q++)
            for (int x = 0; x < 2; x++) again[x] |= order[q][x] == order[p][x];
        if (!again[1]) next_b(order[p][1]);
        if (!again[0]) next_a(order[p][0]);
    }
#pragma unroll
    for (int j = 0; j < FN; j++) {
        tile[j] += sum[j];
        asm volatile("" : "+v"(tile[j]));          // here, not behind the next branch with the sums of a whole step kept for it
    }
}

// C = alpha * op(A) . B + beta * C for one K slice (k_slice a multiple of PK), B from its planes.  A workgroup owns BM x 256 of the
// output; A goes through two LDS buffers in steps of 64 k, one piece of eight k to a thread.  Two groups of eight waves take 32
// k of a step each and add their sums at the end.  BM = 96 and 64: 24573 rows are 256 tiles of 96, one for each compute unit (192
// of 128, with which a quarter of the chip has nothing to do: 90 us), 14000 rows 219 of 64.  part != NULL: the bare product
// of the slice goes to part[slice].  B, ldb: the operand itself, for tiles that are computed again.  Workgroup order as
// sgemm_kernel's.
template <int BM, bool TA, bool TB>
__global__ __launch_bounds__(P_THREADS) void sgemm_planes_kernel(const float *__restrict__ A, int lda,
                                                                 const float *__restrict__ B, int ldb, float *C, int ldc,
                                                                 int M, int N, int K, int k_slice, int tiles_n, int tiles,
                                                                 float alpha, float beta, float *__restrict__ part,
                                                                 const char *__restrict__ planes,
                                                                 const int *__restrict__ inexact, int plane_steps) {
    typedef PlaneOperand<BM, !TA> OpA;
    constexpr int FM = BM / 16, FN = 2, HALF = FM / 2;
    static_assert(FM % 2 == 0 && FM >= 4, "two groups share the fragments; the split goes between two pairs");
    __shared__ __align__(16) char lds[2][OpA::BYTES];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int slice = logical / tiles, tile = logical - slice * tiles;
    const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * PN;
    const int k_beg = slice * k_slice, k_end = min(K, k_beg + k_slice);
    const int steps = (k_end - k_beg) / PK, rest = (k_end - k_beg) % PK, all = steps + (rest > 0);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;
    const int group = wave / (PN / 32), wn = wave % (PN / 32) * 32;
    const bool loads = wave < OpA::PIECES / 64;          // the wave has pieces of A

    v4f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    unsigned left = 0;
    OpA oa;
    oa.start(A, lda, m0, M, k_beg);
    // A step with fewer than PK values of k, the last ones, is taken first: all that are loaded in the loop are whole.
    // the wave's units of B
    const char *pb = planes + ((size_t)((n0 + wn) >> 5) * plane_steps + (k_beg >> 5) + group) * P_UNIT;
    const unsigned lane16 = lane * 16;
    bf8_t a[3], b[FN][3];               // a fragment of A, the wave's two of B
    auto load_b = [&](const char *from, int q) {
#pragma unroll
        for (int j = 0; j < FN; j++) b[j][q] = *reinterpret_cast<const bf8_t *>(from + (3 * j + q) * P_FRAG + lane16);
    };
    const int frag_a = group * (FM * 3 * P_FRAG) + OpA::slot(group, quarter, li);
    auto read_a = [&](const char *buf, int i, int q) {
        a[q] = *reinterpret_cast<const bf8_t *>(buf + frag_a + (i * 3 + q) * P_FRAG);
    };
    if (all > 0) {
        if (rest) {
            oa.fetch_short(steps, rest);
        } else {
            oa.fetch();
            oa.base += steps > 1 ? oa.ahead : 0;
        }
        const char *first = pb + (rest ? (size_t)steps * (2 * P_UNIT) : 0);
#pragma unroll
        for (int q = 0; q < 3; q++) load_b(first, q);
        if (!rest) pb += 2 * P_UNIT;
        if (loads) {
            Planes o;
            split_eight(oa.r, 0, 4, o, left);
            if (steps > 0) oa.fetch();
            oa.write(o, lds[0]);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 3; q++) read_a(lds[0], 0, q);
    }
    // Loads come back in the order they are asked for, and a wait for one is a wait for all before it: the next step's
    // fragments of B, which come from the L2, are asked for ahead of the piece of A of the step after it, which comes from memory.
    // (The step behind the last is the last again: no condition, so that the compiler can count the loads in flight.)
    auto step = [&](auto last_step, int t) __attribute__((always_inline)) {
        constexpr bool more = !decltype(last_step)::value;
        const char *cur = lds[t & 1];
        char *next = lds[(t + 1) & 1];
        auto fragment = [&](auto turn, int i) __attribute__((always_inline)) {
            constexpr Turn TURN = decltype(turn)::value;
            constexpr bool last = TURN == Turn::LAST;
            if (last && more) {
                if (loads) {
                    Planes o;
                    split_eight(oa.r, 0, 4, o, left);
                    oa.write(o, next);
                }
                __syncthreads();                // the tile is in registers, the next one in LDS
            }
            plane_products<TURN, FN>(
                acc[i], a, b, [&](int q) { if (!last || more) read_a(last ? next : cur, last ? 0 : i + 1, q); },
                [&](int q) { if (last && more) load_b(pb, q); });
            __builtin_amdgcn_sched_barrier(0);
        };
        fragment(std::integral_constant<Turn, Turn::FIRST>(), 0);
#pragma unroll
        for (int i = 1; i + 1 < FM; i++) fragment(std::integral_constant<Turn, Turn::MIDDLE>(), i);
        fragment(std::integral_constant<Turn, Turn::LAST>(), FM - 1);
        if (more) {
            pb += 2 * P_UNIT;
            oa.base += t + 2 < all ? oa.ahead : 0;
            if (loads) oa.fetch();
        }
    };
    int t = 0;
    for (; t + 1 < all; t++) step(std::false_type(), t);
    if (t < all) step(std::true_type(), t);

    // The groups' sums: the first half of the rows is finished by the first group, the other by the second.
    typedef v4f Half[HALF][FN];
    static_assert(HALF * FN * 8 * 64 * 16 <= (int)sizeof(lds), "half of the sums fits the buffers");
    v4f *x = reinterpret_cast<v4f *>(&lds[0][0]) + (wave % (PN / 32)) * (HALF * FN * 64) + lane;
    Half half;
#pragma unroll
    for (int g = 0; g < 2; g++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < HALF; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
                if (group != g) x[(i * FN + j) * 64] = acc[g * HALF + i][j];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < HALF; i++)
#pragma unroll
            for (int j = 0; j < FN; j++)
                if (group == g) half[i][j] = acc[g * HALF + i][j] + x[(i * FN + j) * 64];
    }
    // what the planes could not hold of the tile's columns and this slice's k
    for (int i = threadIdx.x; i < 2 * all * (PN / 32); i += P_THREADS) {
        const int c = i / (2 * all), s = i - c * 2 * all;
        left |= inexact[(size_t)((n0 >> 5) + c) * plane_steps + (k_beg >> 5) + s];
    }
    split_finish<HALF, FN, TA, TB, true>(half, left, A, lda, B, ldb, C, ldc, M, N, m0 + 16 * HALF * group, n0 + wn, k_beg, k_end,
                                         alpha, beta, part ? part + (size_t)slice * M * N : nullptr);
}

typedef unsigned v2u __attribute__((ext_vector_type(2)));

// C = alpha * op(A) . B + beta * C where a workgroup holds all of k of its rows of A: 16 * FM rows, split once, in LDS
// (K <= R_STEPS(FM) * 32), and walks over `units` units of 32 columns, eight waves in turn.  B comes from its planes as above;
// behind the one barrier the waves have nothing to do with one another, so one multiplies while another waits for
// old values of C or stores.
constexpr int R_THREADS = 1024;
constexpr int R_LDS = 144 * P_FRAG;                            // of the 160 KB of a compute unit
constexpr int R_UNITS = 64 * (R_THREADS / 64);                 // of a workgroup: a bit each to a wave
constexpr int rows_steps(int FM) { return R_LDS / (3 * P_FRAG * FM); }         // most steps of 32 k

template <int FM, bool TA, bool TB>
__global__ __launch_bounds__(R_THREADS) void sgemm_rows_kernel(const float *__restrict__ A, int lda,
                                                                  const float *__restrict__ B, int ldb, float *C, int ldc,
                                                                  int M, int N, int K, int units, int ranges, float alpha,
                                                                  float beta, const char *__restrict__ planes,
                                                                  const int *__restrict__ inexact, int plane_steps) {
    constexpr int FN = 2, BM = 16 * FM;
    __shared__ __align__(16) char lds[R_LDS];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int m0 = logical / ranges * BM;
    const int unit0 = logical % ranges * units, unit1 = min(unit0 + units, (N + 31) / 32);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, quarter = lane >> 4, li = lane & 15;

    auto slot = [](int ks, int q, int r) { return (16 * q + (r ^ (4 * (ks & 3) + q))) * 16; };
    const unsigned lane16 = lane * 16;
    bf8_t b[FN][3];
    auto load_b = [&](const char *from, int q) {
#pragma unroll
        for (int j = 0; j < FN; j++) b[j][q] = *reinterpret_cast<const bf8_t *>(from + (3 * j + q) * P_FRAG + lane16);
    };
    auto unit_at = [&](int u) { return planes + (size_t)min(u, unit1 - 1) * plane_steps * P_UNIT; };
    const char *pb = unit_at(unit0 + wave);
#pragma unroll
    for (int q = 0; q < 3; q++) load_b(pb, q);

    // the rows of A: pieces of eight k, K contiguous along a row, otherwise along k
    unsigned left = 0;
    {
        constexpr int BATCH = 2;
        const int chunks = plane_steps * 4, pieces = BM * chunks;
        for (int p0 = threadIdx.x; p0 < pieces; p0 += BATCH * R_THREADS) {
            float r[BATCH][8];
#pragma unroll
            for (int i = 0; i < BATCH; i++) {
                const int p = min(p0 + i * R_THREADS, pieces - 1);
                const int x = TA ? p % BM : p / chunks, k = 8 * (TA ? p / BM : p % chunks), m = min(m0 + x, M - 1);
                const float *from = TA ? A + (size_t)k * lda + m : A + (size_t)m * lda + k;
                if (k + 8 <= K) {
                    if constexpr (TA) {
#pragma unroll
                        for (int e = 0; e < 8; e++) r[i][e] = from[(size_t)e * lda];
                    } else {
#pragma unroll
                        for (int q = 0; q < 2; q++) {
                            const v4f v = ld4(from + 4 * q);
#pragma unroll
                            for (int e = 0; e < 4; e++) r[i][4 * q + e] = v[e];
                        }
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) r[i][e] = k + e < K ? from[TA ? (size_t)e * lda : (size_t)e] : 0.f;
                }
            }
#pragma unroll
            for (int i = 0; i < BATCH; i++) {
                const int p = p0 + i * R_THREADS;
                if (p >= pieces) break;
                const int x = TA ? p % BM : p / chunks, c = TA ? p / BM : p % chunks;
                Planes o;
                split_eight(r[i], 0, 4, o, left);
                char *to = lds + ((c >> 2) * FM + (x >> 4)) * (3 * P_FRAG) + slot(c >> 2, c & 3, x & 15);
                *reinterpret_cast<v4u *>(to) = o.h;
                *reinterpret_cast<v4u *>(to + P_FRAG) = o.m;
                *reinterpret_cast<v4u *>(to + 2 * P_FRAG) = o.l;
            }
        }
    }
    const bool a_inexact = __syncthreads_or((left & 0xffffu) != 0);

    const bool read = beta != 0.f;                              // beta == 0 does not read C (cblas semantics)
    const auto out = __builtin_amdgcn_make_buffer_rsrc(C + (size_t)m0 * ldc, 0, min(BM, M - m0) * ldc * 4, 0x00020000);
    bf8_t a[3];
    v4f acc[FM][FN];
    auto read_a = [&](int ks, int i, int q) {
        a[q] = *reinterpret_cast<const bf8_t *>(lds + (size_t)ks * (FM * 3 * P_FRAG) + slot(ks, quarter, li) + (i * 3 + q) * P_FRAG);
    };
    // Rows and columns past the end are out of the buffer's range: not read, not written.  The range check compares the vector
    // offset, so the row is part of that; whether the scalar offset counts too is not the same in every description of it.
    // (96 rows of 2^22 columns end below 2^31, and 2^31 and a row more stays below 2^32.)
    auto row = [&](int i, int e) { return (unsigned)((16 * i + e) * ldc) * 4u; };
    auto finish = [&](int u) __attribute__((always_inline)) {
        const int n = u * 32 + FN * li;
        const unsigned at = n + 1 < N ? (unsigned)(4 * quarter * ldc + n) * 4u : 1u << 31;
#pragma unroll
        for (int i = 0; i < FM; i++) {
            v2f c[4];
            if (read) {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    c[e] = __builtin_bit_cast(v2f, __builtin_amdgcn_raw_buffer_load_b64(out, at + row(i, e), 0, 0));
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v2f v = {acc[i][0][e] * alpha, acc[i][1][e] * alpha};
                if (read) v += beta * c[e];
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), out, at + row(i, e), 0, 0);
            }
        }
        if ((N & 1) && u * 32 + 32 > N) {                        // a last column without a neighbour
            const unsigned last = n + 1 == N ? (unsigned)(4 * quarter * ldc + n) * 4u : 1u << 31;
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float v = acc[i][0][e] * alpha;
                    if (read) v += beta * __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(out, last + row(i, e), 0, 0));
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), out, last + row(i, e), 0, 0);
                }
        }
    };
    if (unit0 + wave >= unit1) return;
#pragma unroll
    for (int q = 0; q < 3; q++) read_a(0, 0, q);
    unsigned long long again = 0;
    for (int u = unit0 + wave; u < unit1; u += R_THREADS / 64) {
        const int flag = inexact[(size_t)u * plane_steps + min(lane, plane_steps - 1)];
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        const char *const pb_next = unit_at(u + R_THREADS / 64);
        for (int s = 0; s < plane_steps; s++) {
            const bool end = s + 1 == plane_steps;
            const char *from = end ? pb_next : pb + (size_t)(s + 1) * P_UNIT;
            auto fragment = [&](auto turn, int i) __attribute__((always_inline)) {
                constexpr Turn TURN = decltype(turn)::value;
                constexpr bool last = TURN == Turn::LAST;
                plane_products<TURN, FN>(
                    acc[i], a, b, [&](int q) { read_a(!last ? s : end ? 0 : s + 1, last ? 0 : i + 1, q); },
                    [&](int q) { if (last) load_b(from, q); });
                __builtin_amdgcn_sched_barrier(0);
            };
            fragment(std::integral_constant<Turn, Turn::FIRST>(), 0);
#pragma unroll
            for (int i = 1; i + 1 < FM; i++) fragment(std::integral_constant<Turn, Turn::MIDDLE>(), i);
            fragment(std::integral_constant<Turn, Turn::LAST>(), FM - 1);
        }
        pb = pb_next;
        const bool bad = a_inexact || flag != 0 || split_not_finite<FM, FN>(acc);
        if (__builtin_amdgcn_ballot_w64(bad) != 0) again |= 1ull << ((u - unit0) / (R_THREADS / 64));
        else finish(u);
    }
    // units to be computed again, behind the loop, where they do not cost it registers
    for (int u = unit0 + wave; again; u += R_THREADS / 64, again >>= 1)
        if (again & 1) {
            split_again<FM, FN, TA, TB, true>(acc, A, lda, B, ldb, M, N, m0, u * 32, 0, K);
            finish(u);
        }
}
