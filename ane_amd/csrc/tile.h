// tile.h — register-tile helpers shared by the strided-axis reduction kernels.
#pragma once
#include "common.h"

#include <type_traits>

template <int VEC>
__device__ __forceinline__ void ldv(float (&r)[VEC], const float *p) {
    if constexpr (VEC == 4) {
        v4f t = ld4(p);
        r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
    } else {
        r[0] = *p;
    }
}
// streaming variants: the operand is touched once by this kernel
template <int VEC>
__device__ __forceinline__ void ldv_nt(float (&r)[VEC], const float *p) {
    if constexpr (VEC == 4) {
        v4f t = ld4_nt(p);
        r[0] = t.x; r[1] = t.y; r[2] = t.z; r[3] = t.w;
    } else {
        r[0] = __builtin_nontemporal_load(p);
    }
}
template <int VEC>
__device__ __forceinline__ void stv_nt(float *p, const float (&r)[VEC]) {
    if constexpr (VEC == 4) {
        v4f t = {r[0], r[1], r[2], r[3]};
        st4_nt(p, t);
    } else {
        __builtin_nontemporal_store(r[0], p);
    }
}
template <int VEC>
__device__ __forceinline__ void stv(float *p, const float (&r)[VEC]) {
    if constexpr (VEC == 4) {
        v4f t = {r[0], r[1], r[2], r[3]};
        st4(p, t);
    } else {
        *p = r[0];
    }
}

// The first loads of a tile that one workgroup holds: past the caches where rows are whole 128-byte lines, through them where a line
// that holds the end of one row piece and the start of another is asked for twice.  RMSNorm of cold operands, past the caches
// always / this: bfloat16 [115][768][54] forward 9.0 / 8.1 us, backward 13.2 / 11.5, with the residual 19.3 / 17.5, [64][1024][256]
// 15.4 / 13.8, 25.0 / 22.8, 42.2 / 39.4; fp32 backward [115][768][54] 27.2 / 25.7, [22][1024][147] 18.0 / 16.1.  The other fp32 tiles
// stay past the caches: forward no difference, with the residual [115][768][54] 21.5 / 24.2.
template <typename F>
__device__ __forceinline__ void first_loads(bool lines, F load) {
    if (lines) load(std::true_type());
    else load(std::false_type());
}
template <int VEC, bool LINES>
__device__ __forceinline__ void ldv_first(float (&r)[VEC], const float *p) {
    if constexpr (LINES) ldv_nt<VEC>(r, p);
    else ldv<VEC>(r, p);
}

// The columns of a lane whose strip gives it columns nominal .. nominal+VEC-1 of rows of S columns (S >= VEC).  Where
// the last group of a row is short, its lane takes the last VEC columns of the row instead: the first `dup` of them are
// also its neighbour's.  Both compute such a column from the same values in the same order and store the same bits, so
// every lane keeps whole vector accesses; sums over the columns of a row skip the duplicates.
// Before, such rows (S % 4 != 0; bfloat16: % 8) were read one column per lane by 32 workgroups for [8][768][197]:
// residual + RMSNorm 97 us, RMSNorm backward + residual 138 us; now on the clustered tiles 8.4 and 9.6 us (19 MB and
// 24 MB: as whole rows of that size take).
struct LaneCols {
    int col, dup;
    bool ok;        // the lane has columns at all
    bool ragged;    // some lane of the launch has duplicates (the same for every lane)
};
// Sum of term(j) over the columns of a lane that are its own.  The sum of all of them is formed first and only rows
// with a short group go back for the masked one: the branch is a scalar one, and whole rows pay no select per column
// (with selects the bfloat16 backward of a [16][1024][256] layer took 0.3 us more).
template <int VEC, typename F>
__device__ __forceinline__ float own_sum(const LaneCols &l, F term) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < VEC; j++) s += term(j);
    if (VEC > 1 && l.ragged) {
        s = 0.f;
#pragma unroll
        for (int j = 0; j < VEC; j++) s += j >= l.dup ? term(j) : 0.f;
    }
    return s;
}
template <int VEC>
__device__ __forceinline__ LaneCols lane_cols(int nominal, int S) {
    LaneCols l;
    l.ok = nominal < S;
    l.col = VEC > 1 && l.ok && nominal > S - VEC ? S - VEC : nominal;
    l.dup = nominal - l.col;
    l.ragged = VEC > 1 && S % VEC != 0;
    return l;
}
// The same, where a lane whose strip gives it no columns at all reads the row's last VEC too: every load is in bounds, none
// behind a condition.  All its columns are duplicates (S >= VEC > 1).
template <int VEC, int W>
__device__ __forceinline__ LaneCols lane_cols_inside(int nominal, int S) {
    LaneCols l;
    l.ok = nominal < S;
    l.col = min(nominal, S - VEC);
    l.dup = min(nominal - l.col, VEC);
    l.ragged = S % W != 0;      // strips are W columns wide
    return l;
}
// Whether an operand may be overwritten in place by a kernel that holds whole tiles in registers: a duplicated column
// must not be written by one workgroup before another has read it, so the short group and its neighbour have to lie in
// the same strip of W columns.
static inline bool tail_in_strip(int S, int W, int VEC) { return S % VEC == 0 || S % W >= VEC; }

// ---- bfloat16 storage: values travel as uint16_t bit patterns (the upper half of the fp32 pattern) and are
// widened to fp32 on load, rounded to nearest even on store ----
typedef uint16_t bf16_t;
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v4u_any __attribute__((ext_vector_type(4), aligned(2)));     // at any bfloat16 element of global memory

__device__ __forceinline__ float bf_to_f(unsigned bits16) { return __uint_as_float(bits16 << 16); }
// round to nearest even; NaN stays NaN (quiet bit forced): the conversion instruction of gfx950, one for two
// values (v_cvt_pk_bf16_f32; the same bits as (u + 0x7fff + ((u >> 16) & 1)) >> 16 with NaNs kept, in a seventh
// of the instructions, which is what the bfloat16 tile kernels spend most of their time on)
__device__ __forceinline__ unsigned f2_to_bf2(float lo, float hi) {
    typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
    typedef float f2_t __attribute__((ext_vector_type(2)));
    const f2_t v = {lo, hi};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf2_t));
}
__device__ __forceinline__ unsigned f_to_bf(float f) { return f2_to_bf2(f, 0.f) & 0xffffu; }

// VEC bf16 values -> VEC floats.  VEC = 8: one 128-bit access, element 2j in the low half of word j.
template <int VEC, bool NT>
__device__ __forceinline__ void ldb(float (&r)[VEC], const bf16_t *p) {
    if constexpr (VEC == 8) {
        const v4u_any *q = reinterpret_cast<const v4u_any *>(p);
        const v4u w = NT ? __builtin_nontemporal_load(q) : *q;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            r[2 * j] = bf_to_f(w[j] & 0xffffu);
            r[2 * j + 1] = bf_to_f(w[j] >> 16);
        }
    } else {
        static_assert(VEC == 1, "bf16 rows are read 8 columns or 1 column at a time");
        r[0] = bf_to_f(*p);
    }
}
template <int VEC, bool FAR = false>
__device__ __forceinline__ void stb(bf16_t *p, const float (&r)[VEC]) {
    if constexpr (VEC == 8) {
        v4u w;
#pragma unroll
        for (int j = 0; j < 4; j++) w[j] = f2_to_bf2(r[2 * j], r[2 * j + 1]);
        if constexpr (FAR) st16_far(p, w);
        else __builtin_nontemporal_store(w, reinterpret_cast<v4u_any *>(p));
    } else {
        *p = (bf16_t)f_to_bf(r[0]);
    }
}

// Register tiles keep the bf16 words packed (half the registers of an fp32 tile) and widen them at each use.
template <int VEC> struct RawT { typedef unsigned type; };
template <> struct RawT<8> { typedef v4u type; };
template <int VEC, bool NT>
__device__ __forceinline__ typename RawT<VEC>::type ld_raw(const bf16_t *p) {
    if constexpr (VEC == 8) {
        const v4u_any *q = reinterpret_cast<const v4u_any *>(p);
        return NT ? __builtin_nontemporal_load(q) : *q;
    } else {
        return (unsigned)*p;
    }
}
template <int VEC>
__device__ __forceinline__ void unpack(float (&r)[VEC], const typename RawT<VEC>::type &w) {
    if constexpr (VEC == 8) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            r[2 * j] = bf_to_f(w[j] & 0xffffu);
            r[2 * j + 1] = bf_to_f(w[j] >> 16);
        }
    } else {
        r[0] = bf_to_f(w);
    }
}
// Tells the compiler nothing about the words' contents from here on, so that the widened copies made before a
// reduction are dropped instead of being kept alive across it (they would double the register tile).
template <int VEC>
__device__ __forceinline__ void forget(typename RawT<VEC>::type &w) {
    if constexpr (VEC == 8) {
        unsigned a = w[0], b = w[1], c = w[2], d = w[3];
        asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
        w[0] = a; w[1] = b; w[2] = c; w[3] = d;
    } else {
        asm volatile("" : "+v"(w));
    }
}
template <int VEC>
__device__ __forceinline__ typename RawT<VEC>::type raw_zero() {
    if constexpr (VEC == 8) { v4u z = {0u, 0u, 0u, 0u}; return z; }
    else return 0u;
}

// Sum acc[q][j] over all threads of the block that share the same lane column (tid % LPR).
// Every thread ends with the full per-column totals.  lds: NW*NV*LPR*VEC floats.
// Across the waves a column is added up by one thread, and every thread then reads its totals: with every thread adding up its
// own columns' waves, 32 reads of 16 bytes and 128 additions for the bfloat16 QK-norm backward on 512 threads, that kernel
// took 3.5 us of its 26 for it ([16][24 x 128][256]).
template <int VEC, int LPR, int THREADS, int NV>
__device__ __forceinline__ void strip_reduce(float (&acc)[NV][VEC], float *lds) {
    constexpr int NW = THREADS / 64;
    constexpr int WLPR = LPR < 64 ? LPR : 64;
    constexpr int TOTALS = NV * WLPR * VEC;
#pragma unroll
    for (int q = 0; q < NV; q++)
#pragma unroll
        for (int j = 0; j < VEC; j++) acc[q][j] = wave_sum_stride<WLPR>(acc[q][j]);
    if constexpr (NW > 1) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int lc = threadIdx.x % LPR;
        if (lane < WLPR) {
#pragma unroll
            for (int q = 0; q < NV; q++)
#pragma unroll
                for (int j = 0; j < VEC; j++) lds[((wave * NV + q) * WLPR + lane) * VEC + j] = acc[q][j];
        }
        __syncthreads();
        for (int i = threadIdx.x; i < TOTALS; i += THREADS) {
            float s = 0.f;
#pragma unroll
            for (int wv = 0; wv < NW; wv++) s += lds[wv * TOTALS + i];
            lds[i] = s;                     // (wave 0's place, which nobody else reads before the barrier)
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NV; q++)
#pragma unroll
            for (int j = 0; j < VEC; j++) acc[q][j] = lds[(q * WLPR + (lc & (WLPR - 1))) * VEC + j];
    }
}


// ---- weight-gradient reductions (dw_reduce.hip) -------------------------------------------------
// A backward op writes per-workgroup partial rows part[nrows][C] and submits "out[c] += sum_r part[r][c]".
// Immediately (default) the jobs of one op go out as one launch when the op ends; in deferred mode they
// are queued and reduced together by mi355_dw_flush().
//
// Buffer for `floats` partials of the op that will accumulate into out0 / out1 (either may be NULL).
float *mi355_dw_partials(size_t floats, const float *out0, const float *out1);
int mi355_dw_submit(float *out, const float *part, int nrows, int C);
int mi355_dw_op_end(void);
