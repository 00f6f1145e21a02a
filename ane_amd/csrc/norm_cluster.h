// norm_cluster.h — RMSNorm forward / backward with the channel axis split over a cluster of workgroups.
//
// The register-tile kernels of norm.hip give one workgroup all C rows of a strip of columns, so a tensor of
// [16][1024][256] has work for 256 workgroups only if a strip is 16 columns: 64-byte pieces of 1 KiB rows, the
// access shape that this memory system serves worst.  Here a strip is 64 columns (256-byte pieces) and its C rows
// are shared by `csplit` workgroups (the members of a cluster).  Each member reduces its own rows to per-column
// partial sums, publishes them, reads the other members' partials, and normalises its rows from registers:
// still one pass over HBM, with 4 x the bytes per request and a workgroup on every compute unit.
//
// Exchange without fences.  A release/acquire pair at agent scope writes back and invalidates a whole L2 on
// this part; instead every partial travels as ONE 8-byte relaxed agent-scope atomic {value, tag} (such a store
// is written through to memory, such a load is served from there), and the tag says which launch wrote it:
//   * workgroup number b owns the slots [b][*] and a launch counter cnt[b], which it alone increments, once, at
//     its end.  Its partials of this launch carry the tag cnt[b] + 1.
//   * a consumer reads cnt[p] of every member p of its cluster when it starts (values of the previous launches:
//     kernel boundaries make them visible), and accepts a slot of p only when its tag is cnt[p] + 1.  A slot
//     written by an earlier launch, of this or any other shape or kernel, has a smaller tag.
//   * nothing is cleared between launches and nothing depends on the host, so a recorded graph can be replayed.
// The wait is bounded: after `spin_ticks` of the 100 MHz clock without the tag (members not resident together, a
// device shared with other work) the workgroup computes the other members' partials itself, with the same code in
// the same order, hence the same bits, and every kernel exits.  A member that publishes late, or whose counter
// was read after it finished, only ever makes a consumer fall back; it cannot make it accept a wrong value.
// The sums are combined in member order by every member, so all members of a cluster normalise with identical
// column sums and the result is run-to-run deterministic.
//
// The kernels are written once for both storage types: fp32 (4 columns per lane, strips of 64 columns) and the
// optional bfloat16 storage (8 columns per lane, strips of 128 columns; arithmetic, sums and weights stay fp32).
//
// Reference ops: rmsnorm and rmsnorm_bwd, training/stories_cpu_ops.h:6-53.
#pragma once
#include "cluster_words.h"
#include "common.h"
#include "tile.h"

namespace {

constexpr int CL_LPR = 16;                        // lanes per row piece: 16 x 16 B = 256 B
constexpr int CL_SLOT_STRIDE = XCH_SLOT_STRIDE;   // 8-byte slots per workgroup: two quantities per column
constexpr int CL_MAX_BLOCKS = XCH_MAX_BLOCKS;     // workgroups per launch that the slot area covers
constexpr int CL_MAX_SPLIT = 8;
typedef Mi355Exchange ClusterWs;

// Storage of the activations: the element type in memory, columns per lane (one 128-bit access), the register
// form of such an access (Raw: for bfloat16 the packed words, half the registers of the widened values, widened at
// each use) and the conversions between Raw and fp32.
struct StoreF32 {
    typedef float T;
    typedef v4f Raw;
    static constexpr int VEC = 4;
    static __device__ __forceinline__ Raw load_nt(const T *p) { return ld4_nt(p); }
    static __device__ __forceinline__ Raw load(const T *p) { return ld4(p); }
    static __device__ __forceinline__ void store_nt(T *p, Raw r) { st4_nt(p, r); }
    static __device__ __forceinline__ void widen(float (&v)[VEC], const Raw &r) { v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w; }
    static __device__ __forceinline__ Raw pack(const float (&v)[VEC]) { Raw r = {v[0], v[1], v[2], v[3]}; return r; }
    static __device__ __forceinline__ Raw zero() { Raw r = {0.f, 0.f, 0.f, 0.f}; return r; }
    static __device__ __forceinline__ void forget(Raw &) {}
};
struct StoreBf16 {
    typedef bf16_t T;
    typedef v4u Raw;
    static constexpr int VEC = 8;
    static __device__ __forceinline__ Raw load_nt(const T *p) { return ld_raw<VEC, true>(p); }
    static __device__ __forceinline__ Raw load(const T *p) { return ld_raw<VEC, false>(p); }
    static __device__ __forceinline__ void store_nt(T *p, Raw r) { __builtin_nontemporal_store(r, reinterpret_cast<v4u_any *>(p)); }
    static __device__ __forceinline__ void widen(float (&v)[VEC], const Raw &r) { unpack<VEC>(v, r); }
    static __device__ __forceinline__ Raw pack(const float (&v)[VEC]) {
        Raw r;
#pragma unroll
        for (int j = 0; j < 4; j++) r[j] = f2_to_bf2(v[2 * j], v[2 * j + 1]);
        return r;
    }
    static __device__ __forceinline__ Raw zero() { return raw_zero<VEC>(); }
    // the widened copies made for the column sums are dropped instead of being kept alive across the exchange
    static __device__ __forceinline__ void forget(Raw &r) { ::forget<VEC>(r); }
};
static_assert(CL_SLOT_STRIDE >= 2 * CL_LPR * StoreBf16::VEC, "two quantities per column must fit a workgroup's slots");

// The first read of an operand's rows: past the caches where rows are whole 128-byte lines, through them otherwise (first_loads in
// tile.h).  Cold operands, us, past / through: backward of fp32 [16][1024][256] 11.4 / 12.0, [32][1024][256] 23.5 / 25.2, with the
// residual 34.8 / 36.4, [32][768][256] with it 25.6 / 28.0; [22][1024][147] 18.0 / 15.9, [8][768][197] 9.2 / 8.3, with the residual
// 10.3 / 9.2, [115][768][54] with it 21.4 / 22.5 (20.1 of operands that the last-level cache holds); bfloat16 [32][768][256] with the
// residual 17.1 / 19.9, [22][1024][147] 14.4 / 12.6.
// Backward kernels of large tensors are quicker past them all the same, if nothing of their operands is in the last-level cache.  Time
// past them over through them at C = 512 / 768 / 1024: fp32, 8 clusters, 0.98 / 1.01 / 1.03, with the residual 1.02 / 1.05 / 1.07;
// 28 clusters 0.99 / 0.96 / 0.97 and 0.97 / 0.96 / 0.97; 64 clusters 0.95 / 0.94 / 0.94 and 0.95 / 0.96 / 0.96; bfloat16 with the
// residual, 32 clusters 0.98, 64 clusters 0.97 / 0.96 / 0.94.  In a layer the operands of smaller tensors still are: fused fp32
// layer of [8][768][197] (4.8 MB) 70.4 us through, 71.7 past, of [16][1024][100] (6.6 MB) 106.4 and 103.2, of [32][768][100] 117.6
// and 112.3; one call per op [32][768][100] (9.8 MB) 124.5 and 125.6, [12][1024][250] (12.3 MB) 185.3 and 181.2; bfloat16
// [40][1024][100] (8.2 MB) 129.3 and 124.6.
// CL_EXACT: every member holds exactly RPS*RPT rows and every strip is whole; CL_LINES: rows are read past the caches; CL_ANY:
// neither.  (One kernel with the loads written twice behind a branch took 27.9 us for the 25.4 of [32][768][256].)
// CL_FEW, with one of the latter two: the members' rows fill at most half of their tiles.  Then the row steps in which no lane has
// a row are passed over; elsewhere that costs more than it saves.  Backward with the residual, us, loaded all the same / passed
// over: fp32 [1][512][32] 8.4 / 8.0, [8][512][54] 9.3 / 8.8, [16][512][147] 18.0 / 17.3, bfloat16 [4][512][33] 11.6 / 10.9;
// forward, bfloat16 [4][768][33], three quarters full, 6.5 / 6.7.
enum { CL_ANY, CL_LINES, CL_EXACT, CL_FEW };
constexpr bool cl_lines(int whole) { return whole == CL_EXACT || whole % CL_FEW == CL_LINES; }
template <typename ST, int WHOLE>
__device__ __forceinline__ typename ST::Raw cluster_load(const typename ST::T *p) { return cl_lines(WHOLE) ? ST::load_nt(p) : ST::load(p); }

// Per-thread partial sums acc[q][j] (q < NV quantities, j < VEC columns of this lane) -> per-column sums of the
// workgroup in wsum[q*W + column], valid for all threads after the barrier.  lds: NW*NV*W floats.
template <int THREADS, int NV, int VEC>
__device__ __forceinline__ void member_sums(float (&acc)[NV][VEC], float *lds, float *wsum) {
    constexpr int NW = THREADS / 64;
    constexpr int W = CL_LPR * VEC;
#pragma unroll
    for (int q = 0; q < NV; q++)
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[q][j] = wave_sum_stride<CL_LPR>(acc[q][j]);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane < CL_LPR) {
#pragma unroll
        for (int q = 0; q < NV; q++)
#pragma unroll
            for (int j = 0; j < VEC; j++) lds[(wave * NV + q) * W + lane * VEC + j] = acc[q][j];
    }
    __syncthreads();
    if (threadIdx.x < NV * W) {
        const int q = threadIdx.x / W, c = threadIdx.x % W;
        float s = 0.f;
#pragma unroll
        for (int wv = 0; wv < NW; wv++) s += lds[(wv * NV + q) * W + c];
        wsum[threadIdx.x] = s;
    }
    __syncthreads();
}

// The launch counters of the cluster's members, one to a lane, and this workgroup's own.  Asked for ahead of the rows and wanted
// only with the column sums.  (A relaxed atomic load: the compiler leaves it where it stands, an ordinary one moves to where the
// sums are published, a trip to memory that everybody waits for.  As a load behind a condition, with one added to it at once, it
// kept every wave from asking for its rows until it was back.)
struct ClusterTags {
    unsigned lanes;
    int mine;
    __device__ __forceinline__ unsigned of(int m) const { return __builtin_amdgcn_readlane(lanes, m) + 1u; }
    __device__ __forceinline__ unsigned own() const { return of(mine); }
};
__device__ __forceinline__ ClusterTags cluster_tags(unsigned *cnt, int first, int member, int csplit) {
    const int m = min((int)(threadIdx.x & 63), csplit - 1);
    return {__hip_atomic_load(cnt + first + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP), member};
}

// Per-thread partial sums acc[q][j] -> the cluster's sum of quantity q over column c, in thread i = q*W + c < NV*W (the others
// return at once): the waves' sums are added up and published, every other member's are fetched by the same thread, all of them
// in flight together, and added in member order.  false: the bounded wait expired for a member of this column.  lds: NW*NV*W
// floats; a barrier stands between the writes to it and the sums.
// One thread has a sum from here to the end: what is formed of it (a division, a square root) is formed once and handed to the
// lanes behind the next barrier.  With the members' sums handed on and added up again by every lane, and the division and the root
// taken by all sixteen waves, there was a barrier more.  With that, the launch counters (cluster_tags) and the order of the loads,
// us by the trace, before and after: with the residual, bfloat16 [16][1024][256] forward 9.9 and 8.4, backward 12.9 and 10.4, fp32
// [8][768][197] 7.8 and 7.2, 9.8 and 8.2; without, fp32 [16][1024][256] 8.1 and 7.2, 10.8 and 10.5, [1][768][256] 5.7 and 4.8, 6.7 and 5.5.
template <int THREADS, int NV, int VEC>
__device__ __forceinline__ bool cluster_totals(float (&acc)[NV][VEC], float *lds, int blk, int first, int member, int csplit,
                                               unsigned long long *slots, const ClusterTags &tags, int spin_ticks,
                                               float &total) {
    constexpr int NW = THREADS / 64, W = CL_LPR * VEC;
    static_assert(NV * W <= CL_SLOT_STRIDE && NV * W <= THREADS, "a member's column sums must fit its slots");
#pragma unroll
    for (int q = 0; q < NV; q++)
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[q][j] = wave_sum_stride<CL_LPR>(acc[q][j]);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned i = threadIdx.x;
    if (lane < CL_LPR) {
#pragma unroll
        for (int q = 0; q < NV; q++)
#pragma unroll
            for (int j = 0; j < VEC; j++) lds[(wave * NV + q) * W + lane * VEC + j] = acc[q][j];
    }
    __syncthreads();
    if (i >= NV * W) return true;
    float own = 0.f;
#pragma unroll
    for (int wv = 0; wv < NW; wv++) own += lds[wv * NV * W + i];
    auto slot = [&](int b) {
        return (unsigned long long *)((char *)(slots + (size_t)b * CL_SLOT_STRIDE) + i * (unsigned)sizeof(unsigned long long));
    };
    __hip_atomic_store(slot(blk), (unsigned long long)tags.own() << 32 | __float_as_uint(own), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    unsigned long long pk[CL_MAX_SPLIT];
    bool ok = false;
    for (long long t0 = 0;;) {
#pragma unroll
        for (int m = 0; m < CL_MAX_SPLIT; m++)
            pk[m] = __hip_atomic_load(slot(first + min(m, csplit - 1)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (spin_ticks < 0) break;                        // test mode: whatever the slots hold is refused
        ok = true;
#pragma unroll
        for (int m = 0; m < CL_MAX_SPLIT; m++)
            ok = ok & ((min(m, csplit - 1) == member) | ((unsigned)(pk[m] >> 32) == tags.of(min(m, csplit - 1))));
        if (ok) break;
        const long long now = wall_clock64();
        if (t0 == 0) t0 = now;
        if (now - t0 >= (long long)spin_ticks) break;
        __builtin_amdgcn_s_sleep(2);
    }
    total = 0.f;
#pragma unroll
    for (int m = 0; m < CL_MAX_SPLIT; m++)
        if (m < csplit) total += m == member ? own : __uint_as_float((unsigned)pk[m]);
    return ok;
}

static_assert(CL_MAX_BLOCKS < 1 << CL_NBLK_BITS && CL_MAX_SPLIT < 1 << (1 << CL_SPLIT_BITS), "the fields hold their values");
// cluster / strips = cluster * recip >> CL_RECIP: both are below 2^10 (at least two members to a cluster), so that the excess of
// the reciprocal, below strips / 2^CL_RECIP, times the cluster stays below 1
static_assert(CL_MAX_BLOCKS / 2 <= 1 << (CL_RECIP / 2) && CL_MAX_BLOCKS / 2 < 1 << CL_STRIP_BITS, "the reciprocal is exact");
__device__ __forceinline__ ClusterGeo cluster_geo(unsigned wa, unsigned wb) {
    return cluster_of(wa, wb, xcd_remap(blockIdx.x, cluster_nblk(wa)));      // the members of a cluster are neighbours on one XCD
}

// FUSE: y = a + alpha*b is formed first (and stored), and the norm is taken of it — the residual add and the
// RMSNorm that follows it (training/training_dynamic/train.m:460-461).  Otherwise x = a and b, y_res are unused.
// WHOLE = CL_EXACT: every member holds exactly RPS*RPT rows and every strip is whole.  Then no row or column needs a mask and
// the loads of the tile are issued back to back without branches, which is worth 0.45 us of the 8 us that the
// forward kernel takes on fp32 [16][1024][256].  In other shapes lanes without a row or without columns load valid ones and
// only their values are dropped, which is still quicker than branches: bfloat16 [5][1024][570] forward 8.0 -> 7.6, with the
// residual 10.7 -> 10.4, backward 12.2 -> 12.0, with it 14.0 -> 13.7; fp32 [115][768][54] with the residual 21.2 -> 20.1.
template <typename ST, int RPT, int THREADS, bool FUSE, int WHOLE>
__global__ __launch_bounds__(THREADS) void rms_fwd_cluster_kernel(const typename ST::T *a, const typename ST::T *b,
                                                                  const float *__restrict__ w, unsigned *cnt, int C, int S,
                                                                  unsigned word_a, unsigned word_b,
                                                                  typename ST::T *__restrict__ yn, typename ST::T *y_res,
                                                                  float alpha, float eps, float invC,
                                                                  unsigned long long *slots, int *fallbacks,
                                                                  int spin_ticks) {
    constexpr bool EXACT = WHOLE == CL_EXACT;
    // sixteen loads ahead of the first use are more than there is room for: [12][1024][500] with the residual 30.9 us, with the branch 28.4
    constexpr bool INSIDE = !(FUSE && RPT == 8 && !EXACT);
    constexpr int VEC = ST::VEC;
    constexpr int W = CL_LPR * VEC;
    constexpr int RPS = THREADS / CL_LPR;
    constexpr int NW = THREADS / 64;
    __shared__ float lds[NW * W];
    __shared__ __align__(16) float col_rr[W];
    __shared__ int failed;
    const ClusterGeo g = cluster_geo(word_a, word_b);
    const int csplit = g.csplit, rows_pm = g.rows_pm;
    const int lc = threadIdx.x % CL_LPR, row0 = threadIdx.x / CL_LPR;
    const LaneCols mine = lane_cols_inside<VEC, W>(g.strip * W + lc * VEC, S);
    const int col = mine.col;
    const bool col_ok = mine.ok;
    const size_t slab_base = (size_t)g.slab * C * S + col;
    const ClusterTags tags = cluster_tags(cnt, g.first, g.member, csplit);

    // rows of member m held by this thread: c = m*rows_pm + row0 + k*RPS, valid while below (m+1)*rows_pm and C
    auto row_of = [&](int m, int k) { return m * rows_pm + row0 + k * RPS; };
    auto row_live = [&](int m, int k) { return row0 + k * RPS < rows_pm && row_of(m, k) < C; };
    auto row_ok = [&](int m, int k) { return row_live(m, k) && col_ok; };
    // one row piece of x (FUSE: of y = a + alpha*b, rounded to the storage type as the stored y is)
    auto sum_row = [&](const typename ST::Raw &ra, const typename ST::Raw &rb) -> typename ST::Raw {
        float av[VEC], bv[VEC], v[VEC];
        ST::widen(av, ra);
        ST::widen(bv, rb);
#pragma unroll
        for (int j = 0; j < VEC; j++) v[j] = bv[j] * alpha + av[j];
        return ST::pack(v);
    };
    auto load_row = [&](int c, bool first) -> typename ST::Raw {
        const size_t off = slab_base + (size_t)c * S;
        const typename ST::Raw ra = first ? cluster_load<ST, WHOLE>(a + off) : ST::load(a + off);
        if constexpr (FUSE) return sum_row(ra, first ? cluster_load<ST, WHOLE>(b + off) : ST::load(b + off));
        else return ra;
    };

    typename ST::Raw xr[RPT], br[FUSE && INSIDE ? RPT : 1];
    float wv[RPT];
    if constexpr (INSIDE) {
        // every load first, then what depends on one: a use between them would wait for it with the others not yet asked for
        auto row = [&](int k) { return EXACT || row_live(g.member, k) ? row_of(g.member, k) : 0; };
        auto none = [&](int k) { return WHOLE >= CL_FEW && k * RPS >= rows_pm; };
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            xr[k] = ST::zero();
            if constexpr (FUSE) br[k] = ST::zero();
            if (none(k)) continue;
            const size_t off = slab_base + (size_t)row(k) * S;
            xr[k] = cluster_load<ST, WHOLE>(a + off);
            if constexpr (FUSE) br[k] = cluster_load<ST, WHOLE>(b + off);
        }
#pragma unroll
        for (int k = 0; k < RPT; k++) wv[k] = w[row(k)];
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            if constexpr (FUSE) xr[k] = sum_row(xr[k], br[k]);
            if (!EXACT && !row_live(g.member, k)) xr[k] = ST::zero();
        }
    } else {
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            if (!row_ok(g.member, k)) {
                xr[k] = ST::zero();
                wv[k] = 0.f;
                continue;
            }
            const int c = row_of(g.member, k);
            xr[k] = load_row(c, true);
            wv[k] = w[c];
        }
    }
    if (threadIdx.x == 0) failed = 0;
    float acc[1][VEC];
#pragma unroll
    for (int j = 0; j < VEC; j++) acc[0][j] = 0.f;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        float xv[VEC];
        ST::widen(xv, xr[k]);
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[0][j] += xv[j] * xv[j];
    }
#pragma unroll
    for (int k = 0; k < RPT; k++) ST::forget(xr[k]);
    float total = 0.f, rr[VEC];
    const bool met = cluster_totals<THREADS, 1, VEC>(acc, lds, g.blk, g.first, g.member, csplit, slots, tags, spin_ticks, total);
    auto scale = [&](float ss) { return 1.0f / sqrtf(ss * invC + eps); };
    if constexpr (FUSE) {
        // the residual goes out while the waves that hold the column sums wait for their partners' (no member that would have to read
        // its rows again finds them overwritten: calls in place take other kernels): odd layer of [8][768][197] 64.4 -> 63.8 us
#pragma unroll
        for (int k = 0; k < RPT; k++)
            if (EXACT || row_ok(g.member, k)) ST::store_nt(y_res + slab_base + (size_t)row_of(g.member, k) * S, xr[k]);
    }
    if (threadIdx.x < W) {
        col_rr[threadIdx.x] = scale(total);
        if (!met) failed = 1;
    }
    __syncthreads();
    if (!failed) {
#pragma unroll
        for (int j = 0; j < VEC; j++) rr[j] = col_rr[lc * VEC + j];
    } else {
        __shared__ float wsum[W];
        float ss[VEC];
#pragma unroll
        for (int j = 0; j < VEC; j++) ss[j] = 0.f;
        if (threadIdx.x == 0) atomicAdd(fallbacks, 1);
        for (int m = 0; m < csplit; m++) {
            float a2[1][VEC];
#pragma unroll
            for (int j = 0; j < VEC; j++) a2[0][j] = 0.f;
#pragma unroll
            for (int k = 0; k < RPT; k++) {
                if (row_ok(m, k)) {
                    float t[VEC];
                    ST::widen(t, load_row(row_of(m, k), false));
#pragma unroll
                    for (int j = 0; j < VEC; j++) a2[0][j] += t[j] * t[j];
                }
            }
            member_sums<THREADS, 1, VEC>(a2, lds, wsum);
#pragma unroll
            for (int j = 0; j < VEC; j++) ss[j] += wsum[lc * VEC + j];
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < VEC; j++) rr[j] = scale(ss[j]);
    }
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        if (EXACT || row_ok(g.member, k)) {
            const size_t off = slab_base + (size_t)row_of(g.member, k) * S;
            float xv[VEC], o[VEC];
            ST::widen(xv, xr[k]);
#pragma unroll
            for (int j = 0; j < VEC; j++) o[j] = (xv[j] * rr[j]) * wv[k];
            ST::store_nt(yn + off, ST::pack(o));
        }
    }
    if (threadIdx.x == 0) cnt[g.blk] = tags.own();
}

// RES: dx = rmsnorm_bwd(dy, x, w) + res and optionally dx2 = alpha2*dx (training/training_dynamic/train.m:586-595,
// :714-721), as rms_bwd_res_kernel of norm.hip.  dw partials: part[cluster][c], one row per cluster.
template <typename ST, int RPT, int THREADS, bool RES, int WHOLE>
__global__ __launch_bounds__(THREADS) void rms_bwd_cluster_kernel(const typename ST::T *__restrict__ x,
                                                                  const typename ST::T *dy, const float *__restrict__ w,
                                                                  unsigned *cnt, int C, int S, unsigned word_a,
                                                                  unsigned word_b, const typename ST::T *res,
                                                                  typename ST::T *dx, float *__restrict__ dw_part,
                                                                  typename ST::T *dx2, float alpha2, float eps, float invC,
                                                                  int variant, unsigned long long *slots, int *fallbacks,
                                                                  int spin_ticks) {
    // without the residual, rows of whole lines keep the branch: [4][768][256] 8.1 us with it, 8.6 without ([8][768][256] with the
    // residual 10.0 and 9.1)
    constexpr bool EXACT = WHOLE == CL_EXACT;
    constexpr bool INSIDE = RES || EXACT || !cl_lines(WHOLE);
    constexpr int VEC = ST::VEC;
    constexpr int W = CL_LPR * VEC;
    constexpr int RPS = THREADS / CL_LPR;
    constexpr int NW = THREADS / 64;
    __shared__ float lds[NW * 2 * W];
    __shared__ __align__(16) float cols[2 * W];      // 1 / rms, then sum (dy*x)*w
    __shared__ int failed;
    const ClusterGeo g = cluster_geo(word_a, word_b);
    const int csplit = g.csplit, rows_pm = g.rows_pm;
    const int lc = threadIdx.x % CL_LPR, row0 = threadIdx.x / CL_LPR;
    const LaneCols mine = lane_cols_inside<VEC, W>(g.strip * W + lc * VEC, S);
    const int col = mine.col;
    const bool col_ok = mine.ok;
    const size_t slab_base = (size_t)g.slab * C * S + col;
    const ClusterTags tags = cluster_tags(cnt, g.first, g.member, csplit);

    auto row_of = [&](int m, int k) { return m * rows_pm + row0 + k * RPS; };
    auto row_live = [&](int m, int k) { return row0 + k * RPS < rows_pm && row_of(m, k) < C; };
    auto row_ok = [&](int m, int k) { return row_live(m, k) && col_ok; };

    typename ST::Raw xr[RPT], dr[RPT], rr_res[RES ? RPT : 1];
    float wv[RPT];
    if constexpr (INSIDE) {
        // every load first, then what depends on one (as above); the residual, needed last, last
        auto row = [&](int k) { return EXACT || row_live(g.member, k) ? row_of(g.member, k) : 0; };
        auto none = [&](int k) { return WHOLE >= CL_FEW && k * RPS >= rows_pm; };
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            xr[k] = dr[k] = ST::zero();
            if (none(k)) continue;
            const size_t off = slab_base + (size_t)row(k) * S;
            xr[k] = cluster_load<ST, WHOLE>(x + off);
            dr[k] = cluster_load<ST, WHOLE>(dy + off);
        }
#pragma unroll
        for (int k = 0; k < RPT; k++) wv[k] = w[row(k)];
        if constexpr (RES) {
#pragma unroll
            for (int k = 0; k < RPT; k++) {
                rr_res[k] = ST::zero();
                if (!none(k)) rr_res[k] = cluster_load<ST, WHOLE>(res + slab_base + (size_t)row(k) * S);
            }
        }
#pragma unroll
        for (int k = 0; k < RPT; k++)
            if (!EXACT && !row_live(g.member, k)) {  // (all three: an infinity in the row read instead would make 0 * inf of the sum)
                xr[k] = dr[k] = ST::zero();
                wv[k] = 0.f;
            }
    } else {
#pragma unroll
        for (int k = 0; k < RPT; k++) {
            xr[k] = dr[k] = ST::zero();
            wv[k] = 0.f;
            if (!row_live(g.member, k)) continue;
            const int c = row_of(g.member, k);
            const size_t off = slab_base + (size_t)c * S;
            xr[k] = cluster_load<ST, WHOLE>(x + off);
            dr[k] = cluster_load<ST, WHOLE>(dy + off);
            wv[k] = w[c];
        }
    }
    if (threadIdx.x == 0) failed = 0;
    float acc[2][VEC];      // [0] = sum x^2, [1] = sum (dy*x)*w
#pragma unroll
    for (int j = 0; j < VEC; j++) acc[0][j] = acc[1][j] = 0.f;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        float xv[VEC], dv[VEC];
        ST::widen(xv, xr[k]);
        ST::widen(dv, dr[k]);
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            acc[0][j] += xv[j] * xv[j];
            acc[1][j] += (dv[j] * xv[j]) * wv[k];
        }
    }
#pragma unroll
    for (int k = 0; k < RPT; k++) { ST::forget(xr[k]); ST::forget(dr[k]); }
    float total = 0.f, rr[VEC], dotn[VEC];
    const bool met = cluster_totals<THREADS, 2, VEC>(acc, lds, g.blk, g.first, g.member, csplit, slots, tags, spin_ticks, total);
    auto scale = [&](float ss) { return 1.0f / sqrtf(ss * invC + eps); };
    auto dot = [&](float sd, float r) { return sd * ((r * r) * invC); };
    if (threadIdx.x < 2 * W) {
        cols[threadIdx.x] = threadIdx.x < W ? scale(total) : total;
        if (!met) failed = 1;
    }
    __syncthreads();
    if (!failed) {
#pragma unroll
        for (int j = 0; j < VEC; j++) {
            rr[j] = cols[lc * VEC + j];
            dotn[j] = dot(cols[W + lc * VEC + j], rr[j]);
        }
    } else {
        __shared__ float wsum[2 * W];
        float ss[VEC], sd[VEC];
#pragma unroll
        for (int j = 0; j < VEC; j++) ss[j] = sd[j] = 0.f;
        if (threadIdx.x == 0) atomicAdd(fallbacks, 1);
        for (int m = 0; m < csplit; m++) {
            float a2[2][VEC];
#pragma unroll
            for (int j = 0; j < VEC; j++) a2[0][j] = a2[1][j] = 0.f;
#pragma unroll
            for (int k = 0; k < RPT; k++) {
                if (row_ok(m, k)) {
                    const size_t off = slab_base + (size_t)row_of(m, k) * S;
                    float tx[VEC], td[VEC];
                    ST::widen(tx, ST::load(x + off));
                    ST::widen(td, ST::load(dy + off));
                    const float wc = w[row_of(m, k)];
#pragma unroll
                    for (int j = 0; j < VEC; j++) {
                        a2[0][j] += tx[j] * tx[j];
                        a2[1][j] += (td[j] * tx[j]) * wc;
                    }
                }
            }
            member_sums<THREADS, 2, VEC>(a2, lds, wsum);
#pragma unroll
            for (int j = 0; j < VEC; j++) { ss[j] += wsum[lc * VEC + j]; sd[j] += wsum[W + lc * VEC + j]; }
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < VEC; j++) { rr[j] = scale(ss[j]); dotn[j] = dot(sd[j], rr[j]); }
    }
    float *part = dw_part + (size_t)(g.first / csplit) * C;
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        const int c = row_of(g.member, k);
        const bool live = EXACT || (row0 + k * RPS < rows_pm && c < C);       // uniform over the 16 lanes of a row piece
        if (live) {
            float xv[VEC], dv[VEC], o[VEC], p = 0.f;
            ST::widen(xv, xr[k]);
            ST::widen(dv, dr[k]);
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                if (variant == 0) o[j] = ((dv[j] - xv[j] * dotn[j]) * rr[j]) * wv[k];
                else o[j] = (dv[j] * wv[k]) * rr[j] - (xv[j] * dotn[j]) * rr[j];
            }
            auto dw_term = [&](int j) { return (dv[j] * xv[j]) * rr[j]; };
            if constexpr (EXACT) {
#pragma unroll
                for (int j = 0; j < VEC; j++) p += dw_term(j);
            } else {
                p = own_sum<VEC>(mine, dw_term);
            }
            if constexpr (RES) {
                float rv[VEC];
                ST::widen(rv, rr_res[k]);
#pragma unroll
                for (int j = 0; j < VEC; j++) o[j] = o[j] + rv[j];
            }
            if (EXACT || col_ok) {
                const size_t off = slab_base + (size_t)c * S;
                ST::store_nt(dx + off, ST::pack(o));
                if constexpr (RES) {
                    if (dx2) {
                        float o2[VEC];
#pragma unroll
                        for (int j = 0; j < VEC; j++) o2[j] = o[j] * alpha2;
                        ST::store_nt(dx2 + off, ST::pack(o2));
                    }
                }
            }
            p = group_sum<CL_LPR>(p);
            if (lc == 0) part[c] = p;
        }
    }
    if (threadIdx.x == 0) cnt[g.blk] = tags.own();
}

// How a shape is split: csplit members of rows_pm rows each; rpt rows per lane.  csplit = 0: not clustered.
struct ClusterPlan {
    int csplit, rows_pm, rpt, threads, strips, nblk;
    int whole;         // which kernel: CL_EXACT, or CL_LINES or CL_ANY, with or without CL_FEW
    unsigned word_a() const { return cluster_word_a(nblk, csplit, rows_pm); }
    unsigned word_b() const { return cluster_word_b(strips); }
};
constexpr ClusterPlan NO_CLUSTER = {0, 0, 0, 0, 0, 0, CL_ANY};

// Clustering pays when whole-C strips of 256 bytes would leave most compute units idle: tall tensors
// (C >= 512) whose strips number fewer than the compute units.  Measured at C = 1024, fp32, with 32 x 256 and
// 64 x 256 columns: a launch of more workgroups than compute units (two rounds of 1024-thread workgroups) loses to
// the single-workgroup tiles with 128-byte strips (forward 30.0 against 29.1 us, backward 22.3 against 19.9 us),
// except for the backward with the residual, whose single-workgroup tile is the weakest (32.7 against 43.7 us).
// vec: columns per lane of the storage type; rpt_lo..rpt_hi: rows per lane that are instantiated (powers of two);
// rounds: how many workgroups per compute unit a launch may have (1: all resident at once).  past: values of a tensor from which on
// rows that are not whole lines are read past the caches as well (cluster_load); 0: never.
ClusterPlan cluster_plan(int C, int S, int batch, bool vec_ok, int vec, int rpt_lo, int rpt_hi, int rounds, size_t past = 0) {
    ClusterPlan p = NO_CLUSTER;
    if (!vec_ok || C < 512 || g_ctx.rms_cluster < 0) return p;
    const int w = CL_LPR * vec;
    const long strips = (long)ceil_div((size_t)S, (size_t)w);
    const long clusters = strips * batch;
    const int cus = g_ctx.num_cu > 0 ? g_ctx.num_cu : 256;
    const int threads = 1024, rps = threads / CL_LPR;
    int split = 0;
    for (int s = 2; s <= CL_MAX_SPLIT; s *= 2) {
        if (clusters * s > CL_MAX_BLOCKS || clusters * s > (long)rounds * cus) break;
        const int rows = (int)ceil_div((size_t)C, (size_t)s);
        if (rows > rps * rpt_hi) continue;                       // does not fit the registers yet: split further
        split = s;
        if (clusters * s >= cus) break;                          // a workgroup for every compute unit
    }
    if (g_ctx.rms_cluster > 0) split = g_ctx.rms_cluster;        // forced (2, 4 or 8) for experiments and tests
    if (split < 2 || split > CL_MAX_SPLIT || (split & (split - 1)) || clusters * split > CL_MAX_BLOCKS) return p;
    const int rows = (int)ceil_div((size_t)C, (size_t)split);
    int rpt = rpt_lo;
    while (rpt < rpt_hi && rows > rps * rpt) rpt *= 2;
    if (rows > rps * rpt) return p;
    p.csplit = split;
    p.rows_pm = rows;
    p.rpt = rpt;
    p.threads = threads;
    p.strips = (int)strips;
    p.nblk = (int)(clusters * split);
    const bool read_past = past > 0 && clusters >= 24 && (size_t)C * S * batch >= past;
    p.whole = rows == rps * rpt && rows * split == C && S % w == 0
                  ? CL_EXACT
                  : (S % (w / 2) == 0 || read_past ? CL_LINES : CL_ANY) + (2 * rows <= rps * rpt ? CL_FEW : 0);
    return p;
}
// (a tile of more than the fewest rows per lane is at least half full: no CL_FEW there)
template <typename F>
void cluster_whole(const ClusterPlan &p, F as) {
    if (p.whole == CL_EXACT) as(std::integral_constant<int, CL_EXACT>());
    else if (p.whole == CL_LINES) as(std::integral_constant<int, CL_LINES>());
    else if (p.whole == CL_LINES + CL_FEW) as(std::integral_constant<int, CL_LINES + CL_FEW>());
    else if (p.whole == CL_ANY + CL_FEW) as(std::integral_constant<int, CL_ANY + CL_FEW>());
    else as(std::integral_constant<int, CL_ANY>());
}

}   // namespace
