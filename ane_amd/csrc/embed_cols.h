// embed_cols.h — the ordered scatter-add of the embedding backward with the columns of dE dealt out to the workgroups.
// Included by embed.hip inside its unnamed namespace.
//
// embed_backward (training/stories_cpu_ops.h:123-131, training/training_dynamic/cpu_ops.h:158-164) adds dx[:,t] into
// dE[tok_t] for t ascending: every (row, d) sum has one fixed fp32 order, and the columns d are independent of one
// another.  Here a workgroup owns K adjacent columns of dE (K = 3 for D = 768, 4 for D = 1024, on 256 compute units)
// and sees every position: its part of dx is K whole rows of every sequence, contiguous in the channel-first layout,
// so dx is read once, coalesced, by exactly one workgroup, and nothing is copied token-major through memory.  The
// positions are taken in blocks of CB, in order; within a block they are ranked by (token, position), so a token's
// positions form a run of consecutive ranks, and a lane adds a run to dE[token][d] sequentially: acc = dE;
// acc += x[rank] for the ranks ascending; dE = acc.  Blocks in ascending order and ranks ascending within a run are
// the order of the reference loop, so the result is that loop's bit for bit.
//
// Two launches (one, col_sum_small_kernel, up to 512 positions):
//   1. block_plan_kernel: 16 to 128 workgroups to a block, each with the tokens of one hash value: rk[position] = its rank within
//      the block, and the block's runs {token, first rank, length}, long runs listed from the front of the block's task
//      array, short ones from its back.
//   2. col_sum_kernel<K>: per block, every thread writes its values of dx (fetched into registers while the previous
//      block was summed) to LDS at their ranks, so that a run is a contiguous piece of an LDS column.  Waves 0..K-1
//      take the long runs of one column each (128-bit LDS reads issued sixteen adds ahead); the other waves take the
//      short runs, K columns to a lane, the old sums of a lane's runs asked for before the block's values are put in
//      their places.  A long run's result also stays in LDS under its token, so the run of the same token in the
//      next block starts from there and not from a load of dE: the chain of the most frequent token, which bounds
//      the whole operation, goes on from block to block without a trip to memory.  The last thing the launch does is
//      to leave the number of runs it saw where the host finds it before the next call (see scatter_form in embed.hip).
#pragma once

constexpr int CB = 8192, CB_BITS = 13;      // positions per block
constexpr int COL_LONG = 16;                // runs of at least this many positions go to the long-run waves
constexpr int COL_CARRY = 256;              // entries of the token-indexed table that carries long runs' sums to the next block
constexpr int COL_PPT = CB / 1024;          // positions of a block per thread
static_assert(COL_PPT % 4 == 0 && CB / 16 / 64 == 8, "values of dx come by fours; a wave of a plan has eight times 64 ids");

typedef unsigned v2u __attribute__((ext_vector_type(2)));

constexpr int PLAN_WORKGROUPS = 256;        // of a plan, over its blocks
constexpr int PLAN_BLOCKS = 64;             // blocks of one pair of launches; more positions are taken in several

// The numbers of long (bits 0 to 15) and short runs (from bit 32) of a block, a line to a block.  Two that take turns: a plan counts in
// one, which the plan before it has cleared, and clears the other.  Bits 16 to 31 count the workgroups that have come with their first
// runs, and the last of them, which all the others have read `turn` before, moves it on.  So nothing is cleared by a launch of
// its own, a recorded graph can be replayed, and a plan leaves a cleared count to the next one whether or not its sums are
// launched (with the turn moved on by the sums, a call that ended between the two left its runs to be counted on top of).
struct __attribute__((aligned(128))) PlanCount {
    unsigned long long runs[2];
    unsigned turn;
};
__device__ PlanCount plan_count[PLAN_BLOCKS];

// v summed over groups of 2^sh adjacent lanes (sh <= 4, the same for all lanes); every lane ends with its group's sum
__device__ __forceinline__ int lanes_sum(int v, int sh) {
    if (sh >= 1) v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);      // quad_perm:[1,0,3,2]
    if (sh >= 2) v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);      // quad_perm:[2,3,0,1]
    if (sh >= 3) v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);     // half of a row mirrored
    if (sh >= 4) v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true);     // a row mirrored
    return v;
}

// Workgroup (block, g) of `groups` to a block ranks the positions whose token falls into group g; ids outside [0, V) count as token V,
// which no run is listed for.  It reads all ids of the block, 512 to a wave: how many fall into the groups before g is its first
// rank; a wave's own go to its list in order of position.  Of 64 of the list the wave finds the equal ones (a comparison with each of the
// first FEW tokens, then a ballot per bit of the others): every distinct token of the 64 is one entry {token, which 64, how many}, and the
// entries (50 to 120, also where one token has a thousand positions) are ranked against all others by counting, 1024 lanes at a time.
// What the sum of the smaller entries' positions is does not depend on their order in LDS.
// Bound by its chain of barriers and trips to memory, no part of which grows with the text; two workgroups fit a compute unit.  In
// place of a launch that sorted chunks of 256 and one that merged them by binary search, us by the trace: 16384 positions of text 12.4,
// now 6.9; 40000 15.3, 7.8 (of which, by the clock: 1 to start and load, 0.6 for the groups, 0.8 for the equal ones, 1.5 for the entries, 1 for the
// counts).  `groups`: as many workgroups as compute units, 128 to a block at most (the first version, in 64 and 32: 7.8 and 9.3).
__global__ __launch_bounds__(1024) void block_plan_kernel(uint16_t *__restrict__ rk, v2u *__restrict__ tasks,
                                                          const int32_t *__restrict__ ids, int N, int V, int key_bits, int groups) {
    constexpr int PER_WAVE = CB / 16, FEW = 12;
    __shared__ __attribute__((aligned(16))) unsigned ent[CB];
    __shared__ unsigned list[CB];                               // PER_WAVE to a wave
    __shared__ uint16_t first_of[1024];
    __shared__ __attribute__((aligned(16))) int wave_less[16];
    __shared__ int n_ent, n_long, n_short, base_long, base_short;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int blk = blockIdx.x / (unsigned)groups;
    const unsigned g = blockIdx.x - blk * groups;
    const int p0 = blk * CB + wave * PER_WAVE + lane;
    int id[PER_WAVE / 64];
#pragma unroll
    for (int j = 0; j < PER_WAVE / 64; j++) id[j] = ids[min(p0 + 64 * j, N - 1)];
    // (an atomic load: it stands where it is, ahead of the counting)
    const unsigned turn = __hip_atomic_load(&plan_count[blk].turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (t == 0) n_ent = n_long = n_short = 0;
    const v4u none = {~0u, ~0u, ~0u, ~0u};                      // behind the entries: not below any
    *reinterpret_cast<v4u *>(&ent[4 * t]) = none;
    *reinterpret_cast<v4u *>(&ent[CB / 2 + 4 * t]) = none;
    __syncthreads();

    unsigned *mine = list + wave * PER_WAVE;
    int n = 0, less = 0;                                        // positions of this wave in group g, and in the groups before it
    const bool whole = (blk + 1) * CB <= N;
#pragma unroll
    for (int j = 0; j < PER_WAVE / 64; j++) {
        const unsigned key = min((unsigned)id[j], (unsigned)V);
        // 16 bits of a product of 24-bit factors, scaled to the number of groups
        unsigned h = (__umul24(__umul24(key, 0x9E3779u) >> 8 & 0xffffu, groups)) >> 16;
        if (!whole && p0 + 64 * j >= N) h = ~0u;
        const unsigned long long owns = __builtin_amdgcn_ballot_w64(h == g);
        if (h == g) mine[n + __builtin_amdgcn_mbcnt_hi((unsigned)(owns >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)owns, 0u))] =
            key << CB_BITS | (unsigned)(wave * PER_WAVE + 64 * j + lane);
        n += __builtin_popcountll(owns);
        less += __builtin_popcountll(__builtin_amdgcn_ballot_w64(h < g));
    }
    if (lane == 0) wave_less[wave] = less;
    for (int c = 0; 64 * c < n; c++) {                          // (a wave's own list: its writes are in order with its reads)
        const int i = 64 * c + lane;
        const bool live = i < n;
        const unsigned w = live ? mine[i] : 0u, k = w >> CB_BITS;
        unsigned long long same = 0, rest = __builtin_amdgcn_ballot_w64(live);
        const unsigned long long all = rest;
        for (int j = 0; j < FEW && rest; j++) {                 // the first tokens one by one: a frequent one is among them
            const unsigned kj = __builtin_amdgcn_readlane(k, __builtin_ctzll(rest));
            const unsigned long long m = __builtin_amdgcn_ballot_w64(k == kj) & all;
            same = k == kj ? m : same;
            rest &= ~m;
        }
        if (rest) {
            unsigned long long eq = rest;
            for (int b = 0; b < key_bits; b++) {
                const unsigned long long ones = __builtin_amdgcn_ballot_w64((k >> b & 1u) != 0);
                const unsigned one = (unsigned)((int)(k << (31 - b)) >> 31);            // all ones where the bit is set
                const unsigned lo = (unsigned)eq & ~((unsigned)ones ^ one), hi = (unsigned)(eq >> 32) & ~((unsigned)(ones >> 32) ^ one);
                eq = (unsigned long long)hi << 32 | lo;
            }
            if (rest >> lane & 1ull) same = eq;
        }
        const int idx = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(same >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)same, 0u));
        const bool head = live && idx == 0;
        const unsigned long long heads = __builtin_amdgcn_ballot_w64(head);
        int e0 = 0;
        if (lane == 0) e0 = atomicAdd(&n_ent, __builtin_popcountll(heads));
        e0 = __builtin_amdgcn_readfirstlane(e0);
        if (live) {
            const int e = e0 + __builtin_popcountll(heads & ((same & -same) - 1ull));       // (the heads ahead of its own)
            if (head) ent[e] = k << CB_BITS | (unsigned)(8 * wave + c) << 6 | (unsigned)(__builtin_popcountll(same) - 1);
            mine[i] = (w & (CB - 1)) | (unsigned)idx << CB_BITS | (unsigned)e << (CB_BITS + 6);
        }
    }
    __syncthreads();

    if (g == 0 && t == 0) plan_count[blk].runs[(turn + 1) & 1] = 0ull;
    const int ne = n_ent;
    const int sh = ne <= 64 ? 4 : ne <= 128 ? 3 : ne <= 256 ? 2 : ne <= 512 ? 1 : 0;       // 2^sh lanes to an entry
    int e1 = 0;
    do {                                                        // (also without an entry: every workgroup counts itself)
        const int e = e1 + (t >> sh), part = t & ((1 << sh) - 1);
        const unsigned w = ent[min(e, CB - 1)], lo = w & ~(CB - 1u), hi = lo + CB;
        int s = 0, upto = 0;                                    // positions of the entries below, and of those up to the token's last
        bool again = false;                                     // the token has an entry below
        if (e < ne)                                             // (the same for the lanes of an entry)
            for (int j = 4 * part; j < ne; j += 4 << sh) {
                const v4u x = *reinterpret_cast<const v4u *>(&ent[j]);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const int m = (int)(x[u] & 63u) + 1;
                    s += x[u] < w ? m : 0;
                    upto += x[u] < hi ? m : 0;
                    again |= x[u] < w && x[u] >= lo;
                }
            }
        s = lanes_sum(s, sh);
        upto = lanes_sum(upto, sh);
        const bool mine_e = e < ne && part == 0, run = lanes_sum(again, sh) == 0 && mine_e && w >> CB_BITS < (unsigned)V;
        const bool is_long = run && upto - s >= COL_LONG;
        if (mine_e) first_of[e - e1] = (uint16_t)s;
        const unsigned long long longs = __builtin_amdgcn_ballot_w64(is_long), shorts = __builtin_amdgcn_ballot_w64(run && !is_long);
        int il = 0, is = 0;
        if (lane == 0 && longs) il = atomicAdd(&n_long, __builtin_popcountll(longs));
        if (lane == 0 && shorts) is = atomicAdd(&n_short, __builtin_popcountll(shorts));
        __syncthreads();
        // the place in the block's lists is a trip to memory; the ranks are written meanwhile
        unsigned long long old = 0;
        if (t == 0 && (n_long | n_short | (e1 == 0)))
            old = atomicAdd(&plan_count[blk].runs[turn & 1],
                            (unsigned long long)(unsigned)n_short << 32 | (e1 == 0 ? 1u << 16 : 0u) | (unsigned)n_long);
        int rank0 = 0;
#pragma unroll
        for (int v = 0; v < 16; v++) rank0 += wave_less[v];
        for (int i = lane; i < n; i += 64) {
            const unsigned x = mine[i];
            const int ex = (int)(x >> (CB_BITS + 6)) - e1;
            if (ex >= 0 && ex < 1024 >> sh)
                rk[(size_t)blk * CB + (x & (CB - 1))] = (uint16_t)(rank0 + first_of[ex] + (x >> CB_BITS & 63u));
        }
        if (t == 0) {
            base_long = (int)(old & 0xffffu);
            base_short = (int)(old >> 32);
            if (e1 == 0 && (int)(old >> 16 & 0xffffu) == groups - 1)
                __hip_atomic_store(&plan_count[blk].turn, turn + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            n_long = n_short = 0;
        }
        __syncthreads();
        il = __builtin_amdgcn_readfirstlane(il);
        is = __builtin_amdgcn_readfirstlane(is);
        if (run) {
            const unsigned long long below = (1ull << lane) - 1ull;
            const int slot = is_long ? base_long + il + __builtin_popcountll(longs & below)
                                     : CB - 1 - (base_short + is + __builtin_popcountll(shorts & below));
            const v2u entry = {w >> CB_BITS, (unsigned)(rank0 + s) | (unsigned)(upto - s) << 16};
            tasks[(size_t)blk * CB + slot] = entry;
        }
        e1 += 1024 >> sh;
    } while (e1 < ne);
}

// acc + x[start] + x[start+1] + ... + x[start+len-1], in that order, from one LDS column.  The column is read in
// aligned groups of eight; what lies outside the run in the first and in the last groups is replaced by -0, which
// leaves every float as it is.  Runs of 32 and more go through a loop of three groups per trip whose reads are
// issued two groups (sixteen adds) ahead of their use, in three register sets that take turns, so the wave issues
// little else than the adds.
__device__ __forceinline__ float long_chain(float acc, const float *xc, int start, int len) {
    const int a0 = start & ~3, lead = start - a0, n = lead + len;       // the run is [lead, n) counted from a0
    const v4f *p = reinterpret_cast<const v4f *>(xc + a0);
    auto add8 = [&](const v4f &c0, const v4f &c1) {
        acc += c0.x; acc += c0.y; acc += c0.z; acc += c0.w;
        acc += c1.x; acc += c1.y; acc += c1.z; acc += c1.w;
    };
    auto masked = [&](const v4f &c0, const v4f &c1, int lo, int hi) {
        acc += (0 >= lo && 0 < hi) ? c0.x : -0.0f; acc += (1 >= lo && 1 < hi) ? c0.y : -0.0f;
        acc += (2 >= lo && 2 < hi) ? c0.z : -0.0f; acc += (3 >= lo && 3 < hi) ? c0.w : -0.0f;
        acc += 4 < hi ? c1.x : -0.0f; acc += 5 < hi ? c1.y : -0.0f;
        acc += 6 < hi ? c1.z : -0.0f; acc += 7 < hi ? c1.w : -0.0f;
    };
    v4f a0_ = p[0], a1_ = p[1];
    masked(a0_, a1_, lead, n);
    int pos = 8;                                                // elements before pos are added
    if (pos + 24 <= n) {
        v4f b0 = p[4], b1 = p[5];                               // group pos + 8
        a0_ = p[2]; a1_ = p[3];                                 // group pos
        v4f c0, c1;
        // at the top: a = group pos, b = group pos + 8, both on their way or here
        for (; pos + 24 <= n; pos += 24) {
            c0 = p[pos / 4 + 4]; c1 = p[pos / 4 + 5];           // group pos + 16
            __builtin_amdgcn_sched_barrier(0);
            add8(a0_, a1_);
            __builtin_amdgcn_sched_barrier(0);
            a0_ = p[pos / 4 + 6]; a1_ = p[pos / 4 + 7];         // group pos + 24
            __builtin_amdgcn_sched_barrier(0);
            add8(b0, b1);
            __builtin_amdgcn_sched_barrier(0);
            b0 = p[pos / 4 + 8]; b1 = p[pos / 4 + 9];           // group pos + 32
            __builtin_amdgcn_sched_barrier(0);
            add8(c0, c1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; pos < n; pos += 8) {                                 // fewer than 24 are left (more for a run that never had 32)
        a0_ = p[pos / 4]; a1_ = p[pos / 4 + 1];
        masked(a0_, a1_, 0, n - pos);
    }
    return acc;
}

// K adjacent floats of a row of dE, moved as one access (4-byte aligned)
template <int K>
struct __attribute__((packed, aligned(4))) ColVec { float f[K]; };

// FULL: D is a multiple of K, every workgroup has K columns.  ANY: sequences of any length, dx at any 4-byte boundary: a
// group of four positions that runs into the next sequence is read one by one (by a lane or two of a wave: at D = 768
// 16351 positions in sequences of 197 take 47 us, the row form 63; 16384 in sequences of 256 take 44); without it S is a
// multiple of 4 and dx 16-byte aligned.
template <int K, bool FULL, bool ANY>
__global__ __launch_bounds__(1024) void col_sum_kernel(float *dE, const float *__restrict__ dx,
                                                       const v2u *__restrict__ tasks,
                                                       const uint16_t *__restrict__ rk, int first, int N, int D, int S, int nblk,
                                                       unsigned long long *report) {
    constexpr int XP = CB + 48;                                 // a column in LDS, with room for the reads issued ahead
    constexpr int NSL = (16 - K) * 64;                          // lanes that take short runs
    constexpr int RPL = 4;                                      // runs of a block whose old sums a lane asks for in one go
    __shared__ __attribute__((aligned(16))) float xs[K][XP];
    __shared__ unsigned long long carry[2][K][COL_CARRY];       // {token, bits of the sum} of the long runs of a block
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int d0 = xcd_remap(blockIdx.x, gridDim.x) * K;        // neighbouring columns on one XCD: they share lines of dE
    const int kv = FULL ? K : min(K, D - d0);                   // columns of this workgroup that exist
    const bool hot = wave < K;                                  // wave d < K: the long runs of column d0 + d
    const int sl = (wave - K) * 64 + lane;                      // the other lanes: short runs, all K columns each

    // a thread's positions in a block, by fours: the loads of a wave are whole lines side by side (eight in a row to a thread, half of
    // every line came with one load and half with the next: 16384 positions into [32000][768] 32.0 us, now 29.4, 40000 into [151936][1024] 88.4, now 75.0)
    auto place = [&](int q) { return 4 * (t + 1024 * q); };
    // What a thread fetches ahead for a block: its positions' values of dx and ranks, the numbers of runs, and the
    // first runs it will take.
    struct Pre {
        v4f px[K][COL_PPT / 4];
        v2u prk[COL_PPT / 4];
        unsigned long long pc;
        v2u pd[RPL];
    };
    Pre o;
    auto fetch_runs = [&](Pre &o, int blk) __attribute__((always_inline)) {
        const v2u *tb = tasks + (size_t)blk * CB;
        const PlanCount c = plan_count[blk];
        o.pc = (c.turn & 1 ? c.runs[0] : c.runs[1]) & ~0xffff0000ull;       // (the plan has moved its turn on)
#pragma unroll
        for (int i = 0; i < RPL; i++) o.pd[i] = tb[hot ? lane + 64 * i : CB - 1 - (sl + NSL * i)];
    };
    auto fetch_values = [&](Pre &o, int blk) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < COL_PPT / 4; q++) {
            const int p0 = first + blk * CB + place(q), p = p0 < N ? p0 : 0;       // (past the end: any address; the values are not used)
            const int b = p / S, s = p - b * S;
            if (!ANY || s + 4 <= S) {
#pragma unroll
                for (int d = 0; d < K; d++)
                    o.px[d][q] = ld4_nt(dx + ((size_t)b * D + d0 + (d < kv ? d : 0)) * S + s);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int pj = p + j < N ? p + j : 0, bj = pj / S;
                    const float *src = dx + ((size_t)bj * D + d0) * S + (pj - bj * S);
#pragma unroll
                    for (int d = 0; d < K; d++) o.px[d][q][j] = src[(size_t)(d < kv ? d : 0) * S];
                }
            }
        }
#pragma unroll
        for (int q = 0; q < COL_PPT / 4; q++) o.prk[q] = *reinterpret_cast<const v2u *>(rk + (size_t)blk * CB + place(q));
    };
    float *dcol = dE + d0 + (hot ? wave : 0);
    const float *xc = &xs[hot ? wave : 0][0];
    const bool col_ok = wave < kv;

    // The long runs of the first block start from dE itself, and the chain of the most frequent token is what the
    // launch waits for.  The waves that take them are the first of the workgroup to issue anything, so their piece of
    // the run list is back within half a microsecond; they ask for their old sums then, ahead of every value of dx,
    // and have them when the block is in its place (asked for with everybody else's, behind 25 MB of dx, they come
    // 2.4 us after that for the median workgroup and 4.8 us for the slowest).
    fetch_runs(o, 0);
    float h0 = 0.f;
    if (hot) {
        const bool hv = col_ok && lane < (int)(o.pc & 0xffffffffu);
        h0 = dcol[(size_t)(hv ? o.pd[0].x : 0u) * D];
    }
    fetch_values(o, 0);
    int runs = 0;
    for (int blk = 0; blk < nblk; blk++) {
        const int n_long = (int)(o.pc & 0xffffffffu), n_short = (int)(o.pc >> 32);
        runs += n_long + n_short;
        const v2u *tb = tasks + (size_t)blk * CB;
        v2u dsc_[RPL];
#pragma unroll
        for (int i = 0; i < RPL; i++) dsc_[i] = o.pd[i];
        __syncthreads();                                    // the previous block's runs are summed and stored
        // the old sums are asked for first: they travel while the block's values are put in their places
        // (every wave issues the same loads, a row that is not needed read as row 0: the wait for the values of
        // dx below then counts these loads exactly and does not include them)
        float acc[RPL][K];
        bool valid[RPL];
        unsigned row[RPL];
        bool hvalid = false, hcarried = false;
        float hacc = 0.f;
#pragma unroll
        for (int i = 0; i < RPL; i++) {
            valid[i] = !hot && sl + NSL * i < n_short;
            row[i] = valid[i] ? dsc_[i].x : 0u;
        }
        if (hot) {
            hvalid = col_ok && lane < n_long;
            const unsigned tok = hvalid ? dsc_[0].x : 0u;
            if (hvalid && blk > 0) {
                const unsigned long long e = carry[(blk - 1) & 1][wave][tok & (COL_CARRY - 1)];
                if ((unsigned)e == tok) {
                    hacc = __uint_as_float((unsigned)(e >> 32));
                    hcarried = true;
                }
            }
            if (blk == 0) {
                hacc = h0;
                hcarried = true;
            }
            row[0] = hvalid && !hcarried ? tok : 0u;
        }
#pragma unroll
        for (int i = 0; i < RPL; i++) {
            const float *src = dE + (size_t)row[i] * D + d0;
            if (FULL || kv == K) {                                  // one request for the K columns
                const ColVec<K> v = *reinterpret_cast<const ColVec<K> *>(src);
#pragma unroll
                for (int d = 0; d < K; d++) acc[i][d] = v.f[d];
            } else {
#pragma unroll
                for (int d = 0; d < K; d++) acc[i][d] = src[d < kv ? d : 0];
            }
        }
#pragma unroll
        for (int q = 0; q < COL_PPT; q++) {
            const int r = (o.prk[q / 4][q / 2 & 1] >> (16 * (q & 1))) & 0xffff;
            if (first + blk * CB + place(q / 4) + (q & 3) < N) {
#pragma unroll
                for (int d = 0; d < K; d++) xs[d][r] = o.px[d][q / 4][q & 3];
            }
        }
        if (t < K * COL_CARRY) carry[blk & 1][t / COL_CARRY][t % COL_CARRY] = ~0ull;
        __syncthreads();
        if (blk + 1 < nblk) {                               // (behind the loads of the old sums: those arrive first)
            fetch_runs(o, blk + 1);
            fetch_values(o, blk + 1);
        }
        // Nobody adds before the next block's values are there: stores to dE and loads of dx disturb each other.  With the loop written
        // so that the sums do not wait (the last block, which fetches nothing, apart), 40000 positions into [151936][1024] took 84 us
        // and 16384 into [32000][768] 36.5, with this 78 and 35.2; with only the long runs' waves not waiting 80.6 and 37.0, with
        // those waves fetching behind their chains 84.5 and 36.1.  (Single positions apart from runs of two and more, so that a
        // wave's stores follow each other without a loop between: 82.9 and 36.8.)
        __builtin_amdgcn_s_waitcnt(0x0f70);                 // vmcnt(0)
        if (hot) {
            __builtin_amdgcn_s_setprio(3);
            if (hvalid) {
                const unsigned tok = dsc_[0].x;
                if (!hcarried) {
#pragma unroll
                    for (int d = 0; d < K; d++)
                        if (d == wave) hacc = acc[0][d];
                }
                hacc = long_chain(hacc, xc, (int)(dsc_[0].y & 0xffffu), (int)(dsc_[0].y >> 16));
                dcol[(size_t)tok * D] = hacc;
                carry[blk & 1][wave][tok & (COL_CARRY - 1)] = ((unsigned long long)__float_as_uint(hacc) << 32) | tok;
            }
            for (int r = 1; r * 64 < n_long; r++) {          // more than 64 long runs in the block
                const int a = lane + 64 * r;
                const bool val = col_ok && a < n_long;
                const v2u dsc = tb[min(a, CB - 1)];
                const unsigned tok = val ? dsc.x : 0u;
                float ac = 0.f;
                bool need = val;
                if (val && blk > 0) {
                    const unsigned long long e = carry[(blk - 1) & 1][wave][tok & (COL_CARRY - 1)];
                    if ((unsigned)e == tok) {
                        ac = __uint_as_float((unsigned)(e >> 32));
                        need = false;
                    }
                }
                if (need) ac = dcol[(size_t)tok * D];
                if (val) {
                    ac = long_chain(ac, xc, (int)(dsc.y & 0xffffu), (int)(dsc.y >> 16));
                    dcol[(size_t)tok * D] = ac;
                    carry[blk & 1][wave][tok & (COL_CARRY - 1)] = ((unsigned long long)__float_as_uint(ac) << 32) | tok;
                }
            }
            __builtin_amdgcn_s_setprio(0);
        } else {
            auto finish = [&](const v2u dsc, float (&ac)[K]) {
                const int start = (int)(dsc.y & 0xffffu), len = (int)(dsc.y >> 16);
#pragma unroll 4
                for (int jj = 0; jj < len; jj++) {
#pragma unroll
                    for (int d = 0; d < K; d++) ac[d] += xs[d][start + jj];
                }
                float *dst = dE + (size_t)dsc.x * D + d0;
                if (FULL || kv == K) {
                    ColVec<K> v;
#pragma unroll
                    for (int d = 0; d < K; d++) v.f[d] = ac[d];
                    *reinterpret_cast<ColVec<K> *>(dst) = v;
                } else {
#pragma unroll
                    for (int d = 0; d < K; d++)
                        if (d < kv) dst[d] = ac[d];
                }
            };
#pragma unroll
            for (int i = 0; i < RPL; i++)
                if (valid[i]) finish(dsc_[i], acc[i]);
            for (int r0 = RPL; r0 * NSL < n_short; r0++) {   // more short runs than RPL per lane: one at a time
                const int s = sl + r0 * NSL;
                if (s >= n_short) continue;
                const v2u dsc = tb[CB - 1 - s];
                const float *src = dE + (size_t)dsc.x * D + d0;
                float ac[K];
#pragma unroll
                for (int d = 0; d < K; d++) ac[d] = src[d < kv ? d : 0];
                finish(dsc, ac);
            }
        }
    }
    // what the host looks at before it picks a form for the next call of this shape (one 8-byte store to host memory)
    if (report && blockIdx.x == 0 && t == 0) *report = scatter_report(runs, N, D, 1);
}

// Up to COL_SMALL positions (one sequence of the reference's loops): plan and sums in ONE launch.  Every workgroup
// ranks all positions itself in LDS (two threads per position count the smaller words; 1 us, redundant but without
// a launch boundary), marks the first rank of every run in a 512-bit mask, writes its K columns of dx to LDS at their
// ranks and sums the runs, one lane per (run, column), from dE and back to it.  Any S.
constexpr int COL_SMALL = 512, COL_SMALL_BITS = 10;

template <int K>
__global__ __launch_bounds__(1024) void col_sum_small_kernel(float *dE, const float *__restrict__ dx,
                                                             const int32_t *__restrict__ ids, int N, int V, int D, int S) {
    constexpr int XP = COL_SMALL + 48;
    __shared__ __attribute__((aligned(16))) unsigned words[COL_SMALL];
    __shared__ unsigned sorted[COL_SMALL];
    __shared__ unsigned short rank_of[COL_SMALL];
    __shared__ unsigned long long heads[COL_SMALL / 64];
    __shared__ __attribute__((aligned(16))) float xs[K][XP];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int d0 = xcd_remap(blockIdx.x, gridDim.x) * K;
    const int kv = min(K, D - d0);
    // this thread's values of dx: element i = column i / N, position i % N (coalesced along the positions)
    constexpr int XPT = (COL_SMALL * K + 1023) / 1024;
    float xv[XPT];
#pragma unroll
    for (int q = 0; q < XPT; q++) {
        const int i = t + 1024 * q, d = i / N, p = i - d * N;
        xv[q] = 0.f;
        if (d < kv) {
            const int b = p / S;
            xv[q] = dx[((size_t)b * D + d0 + d) * S + (p - b * S)];
        }
    }
    if (t < COL_SMALL) {
        unsigned key = (unsigned)V;                             // padding and out-of-range ids sort last
        if (t < N) {
            const int id = ids[t];
            if (id >= 0 && id < V) key = (unsigned)id;
        }
        words[t] = (key << COL_SMALL_BITS) | (unsigned)t;
    }
    __syncthreads();
    {
        const int p = t >> 1, h = t & 1;
        const unsigned w = words[p];
        int r = 0;
#pragma unroll 8
        for (int j = 0; j < COL_SMALL / 2; j += 4) {
            const v4u q = *reinterpret_cast<const v4u *>(&words[h * (COL_SMALL / 2) + j]);
            r += (q.x < w ? 1 : 0) + (q.y < w ? 1 : 0) + (q.z < w ? 1 : 0) + (q.w < w ? 1 : 0);
        }
        r += __shfl_xor(r, 1, 64);
        if (h == 0) {
            rank_of[p] = (unsigned short)r;
            sorted[r] = w;
        }
    }
    __syncthreads();
    if (t < COL_SMALL) {
        // a run starts where the token changes; the first padding word starts one too, so every run ends at a mark
        const bool head = t == 0 || (sorted[t - 1] >> COL_SMALL_BITS) != (sorted[t] >> COL_SMALL_BITS);
        const unsigned long long m = __builtin_amdgcn_ballot_w64(head);
        if (lane == 0) heads[wave] = m;
    }
#pragma unroll
    for (int q = 0; q < XPT; q++) {
        const int i = t + 1024 * q, d = i / N, p = i - d * N;
        if (d < K) xs[d][rank_of[p]] = xv[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < XPT; q++) {
        const int i = t + 1024 * q, d = i / COL_SMALL, r = i % COL_SMALL;
        const unsigned tok = sorted[r] >> COL_SMALL_BITS;
        const bool head = (heads[r >> 6] >> (r & 63)) & 1ull;
        if (d < kv && head && tok < (unsigned)V) {
            // the next mark after r
            int end = COL_SMALL;
            unsigned long long m = (r & 63) == 63 ? 0ull : (heads[r >> 6] >> ((r & 63) + 1));
            if (m) end = r + 1 + __builtin_ctzll(m);
            else
                for (int wq = (r >> 6) + 1; wq < COL_SMALL / 64; wq++)
                    if (heads[wq]) { end = wq * 64 + __builtin_ctzll(heads[wq]); break; }
            float *dst = dE + (size_t)tok * D + d0 + d;
            *dst = long_chain(*dst, &xs[d][0], r, end - r);
        }
    }
}

// Columns of dE per workgroup: three from D = 513 on (256 workgroups at D = 768), four from 769 (256 at D = 1024:
// 148 KB of LDS, the most a workgroup can hold of a block of 8192 positions).
int cols_per_workgroup(int D) { return D > 768 ? 4 : D > 512 ? 3 : D > 256 ? 2 : 1; }

// Launches the kernels of the column form.  The caller has checked V < 2^(32 - CB_BITS).
int scatter_add_cols(float *dE, const float *dx, const int32_t *ids, int V, int D, int S, int N,
                     unsigned long long *report) {
    const int K = cols_per_workgroup(D);
    const dim3 grid((unsigned)ceil_div((size_t)D, K));
    if (N <= COL_SMALL) {
#define COL_LAUNCH(KK)                                                                                              \
    case KK:                                                                                                        \
        hipLaunchKernelGGL(col_sum_small_kernel<KK>, grid, dim3(1024), 0, g_ctx.stream, dE, dx, ids, N, V, D, S);   \
        break;
        switch (K) { COL_LAUNCH(1) COL_LAUNCH(2) COL_LAUNCH(3) COL_LAUNCH(4) }
#undef COL_LAUNCH
        LAUNCH_OK("embed_scatter_add column sums");
        return 0;
    }
    constexpr int MOST = PLAN_BLOCKS * CB;
    const int most_blocks = (int)ceil_div((size_t)std::min(N, MOST), CB);
    size_t total = 0;
    auto take = [&total](size_t bytes) {
        const size_t off = total;
        total += (bytes + 255) & ~(size_t)255;
        return off;
    };
    const size_t off_rk = take((size_t)most_blocks * CB * sizeof(uint16_t));
    const size_t off_tasks = take((size_t)most_blocks * CB * sizeof(v2u));
    char *ws = (char *)mi355_ws(total);
    if (!ws) return -1;
    uint16_t *rk = (uint16_t *)(ws + off_rk);
    v2u *tasks = (v2u *)(ws + off_tasks);
    const bool any = S % 4 != 0 || !aligned16(dx);
    for (int first = 0; first < N; first += std::min(MOST, N - first)) {
        const int n = std::min(MOST, N - first), nblk = (int)ceil_div((size_t)n, CB);
        const int groups = std::max(16, std::min(128, PLAN_WORKGROUPS / nblk));
        hipLaunchKernelGGL(block_plan_kernel, dim3(nblk * groups), dim3(1024), 0, g_ctx.stream, rk, tasks, ids + first, n, V,
                           32 - __builtin_clz((unsigned)V), groups);
        LAUNCH_OK("embed_scatter_add plan");
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(1024), 0, g_ctx.stream, dE, dx, tasks, rk, first, N, D, S, nblk, report);
        };
#define COL_LAUNCH(KK)                                                     \
    case KK:                                                               \
        if (D % KK == 0 && !any) launch(col_sum_kernel<KK, true, false>);  \
        else if (D % KK == 0) launch(col_sum_kernel<KK, true, true>);      \
        else if (!any) launch(col_sum_kernel<KK, false, false>);           \
        else launch(col_sum_kernel<KK, false, true>);                      \
        break;
        switch (K) {
            COL_LAUNCH(1) COL_LAUNCH(2) COL_LAUNCH(3) COL_LAUNCH(4)
        default: return mi355_fail("embed_scatter_add: no kernel for %d columns per workgroup", K);
        }
#undef COL_LAUNCH
        LAUNCH_OK("embed_scatter_add column sums");
    }
    return 0;
}
