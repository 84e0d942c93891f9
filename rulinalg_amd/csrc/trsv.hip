// Triangular solves on nrhs right-hand sides (vector r at in + r * ldi),
// one launch per step of TSB x 64 rows.
//
// A step owns the rows [s0, s1) of one "super-block" (TSB sub-blocks of 64
// rows, taken in solve order).  Every workgroup of the launch first solves
// the super-block redundantly: it stages the super-block's part of the
// triangle in LDS and one wave per right-hand side runs the substitution
// with the vector held in registers (lane i = row i of a sub-block) and the
// solved entry broadcast lane to lane, so no workgroup ever waits for
// another.  Then each workgroup removes the contribution of the solved rows
// from its share of the rows still to be solved (a GEMV slice: rows below
// the super-block for forward substitution, rows above it for backward).
// Workgroup 0 writes the solved rows to `out`.
//
// `in` holds the right-hand sides and is used as the running residual: a
// step reads the rows of its super-block (final since the previous step)
// and updates only rows outside it, so reads and writes of one launch never
// touch the same element.  The solution goes to `out`, a different buffer.
//
// Within a sub-block the entries are found by a column sweep, as in the
// reference's transpose_back_substitution (src/matrix/decomposition/
// cholesky.rs:329-361); forward_substitution, lu_forward_substitution and
// back_substitution (src/matrix/mod.rs:318-398, lu.rs:624-642) form row dot
// products instead; the results agree to rounding.
//
// A launch is bound by its serial chain, 64 columns per sub-block, on top of
// one launch and one memory latency.  So a lane divides its row of the triangle
// and its right-hand side by the row's diagonal up front, which leaves a
// broadcast and one fused multiply-add per column on the chain, and a wave
// sweeps up to four right-hand sides together.  Scaled and swept that way, a
// value that is not finite could reach entries it must not, and a quotient below
// the normal numbers would lose a term; a sub-block whose result holds the one or
// may have lost the other (sweep_lossy) is swept again with a division and a test
// per column.
// FP64 at order 4096, per launch of 128 rows: 14.6 -> 9.1 us (upper, one
// right-hand side), 10.3 -> 8.6 (unit lower); at order 16384 with 16
// right-hand sides 56 -> 17.9 and 39.5 -> 17.2 us.
//
// The loads come next: with a test and a 64-bit product per load, a wave spends
// some 500 instructions before the first barrier.  So no load has a test, and those
// of a whole block are a constant or a scalar apart: solves of order 4096 4 % faster
// (LU 541 -> 520 us, 16 right-hand sides 1,017 -> 980; Cholesky 588 -> 567).
// Taking four entries at a time from the lanes, and their solution redundantly in
// each, is slower (541 -> 594 us): the chain is bound by instructions issued.
#include <limits>

#include "kernels.hpp"
#include "mfma.hpp"
#include "wave.hpp"

namespace rlg {

constexpr int SB = 64;      // sub-block rows (the lanes of one wave)
constexpr int TSB = 2;      // sub-blocks per step
constexpr int TMAXR = 16;   // right-hand sides per launch
constexpr int RPW = 64;     // rows updated per workgroup (row-access forms)
constexpr int CPW = 64;     // entries updated per workgroup (transposed form)

enum TriMode { LOWER_UNIT = 0, LOWER = 1, UPPER = 2, LOWER_T = 3 };

// a / d from r = 1 / d, with one residual correction (Markstein).  Unlike div_recip it
// does not look at the residual: a sub-block with a value that is not finite is swept
// plainly.
template <class T> __device__ __forceinline__ T scaled(T a, T d, T r) {
    const T q = a * r;
    return fma(fma(-q, d, a), r, q);
}

template <int MODE> __device__ __forceinline__ constexpr bool forward() {
    return MODE == LOWER_UNIT || MODE == LOWER;
}
template <int MODE> __device__ __forceinline__ constexpr bool stored_upper() { return MODE == UPPER; }

// One 64 x 64 tile of M (rows rb.., cols cb.., rs x cs valid), 16 values per
// thread: tile_load issues the loads, tile_store puts them in LDS.  `diag`
// keeps only the strict part of the stored triangle and zeroes the rest, so
// entries of the other triangle are never read as numbers.  With `vec` (M and lda allow
// 16-byte loads) a full tile is read with 16-byte loads, a quarter (FP32)
// or half (FP64) of the load instructions: with the update slice also in
// flight, scalar loads would exceed what a wave can have outstanding.
// Staged rows are padded to 16-byte multiples (TP) so that a lane can read
// its row back with 16-byte LDS reads.
constexpr int TPER = SB * SB / 256;
template <class T> constexpr int TVL = 16 / sizeof(T);  // elements per 16 bytes
template <class T> constexpr int TP = TVL<T>;           // row padding
template <class T, int MODE>
__device__ __forceinline__ void tile_load(T (&v)[TPER], const T *__restrict__ M, long lda, int rb,
                                          int cb, int rs, int cs, bool diag, bool vec) {
    constexpr int VL = TVL<T>;
    typedef T vT __attribute__((ext_vector_type(VL)));
    if (vec && rs == SB && cs == SB) {
        constexpr int RPU = 256 / (SB / VL);  // rows per load: their addresses differ by a scalar
        const int i0 = threadIdx.x / (SB / VL), j0 = (threadIdx.x % (SB / VL)) * VL;
        const T *p = M + (long)(rb + i0) * lda + cb + j0;
#pragma unroll
        for (int u = 0; u < TPER / VL; ++u) {
            const int i = u * RPU + i0;
            const vT x = *reinterpret_cast<const vT *>(p + u * (RPU * lda));
#pragma unroll
            for (int t = 0; t < VL; ++t) {
                const int j = j0 + t;
                const bool ok = !diag || (stored_upper<MODE>() ? j > i : j < i);
                v[u * VL + t] = ok ? x[t] : T(0);
            }
        }
    } else {
#pragma unroll
        for (int q = 0; q < TPER; ++q) {
            const int e = q * 256 + threadIdx.x;
            const int i = e >> 6, j = e & 63;
            bool ok = i < rs && j < cs;
            if (diag) ok = ok && (stored_upper<MODE>() ? j > i : j < i);
            v[q] = ok ? M[(long)(rb + i) * lda + cb + j] : T(0);
        }
    }
}
template <class T>
__device__ __forceinline__ void tile_store(T (*tl)[SB + TP<T>], const T (&v)[TPER], bool vec_full) {
    constexpr int VL = TVL<T>;
    if (vec_full) {
#pragma unroll
        for (int u = 0; u < TPER / VL; ++u) {
            const int e = u * 256 + threadIdx.x;
            const int i = e / (SB / VL), j0 = (e % (SB / VL)) * VL;
#pragma unroll
            for (int t = 0; t < VL; ++t) tl[i][j0 + t] = v[u * VL + t];
        }
    } else {
#pragma unroll
        for (int q = 0; q < TPER; ++q) {
            const int e = q * 256 + threadIdx.x;
            tl[e >> 6][e & 63] = v[q];
        }
    }
}

// Row `lane` of a staged tile into registers (r[c] = t[lane][c]), or for the
// transposed form its column `lane` (r[c] = t[c][lane]): the serial chain of
// the substitution then reads registers, not LDS.
template <class T, int MODE>
__device__ __forceinline__ void tile_row(const T (*t)[SB + TP<T>], int lane, T (&r)[SB]) {
    constexpr int VL = TVL<T>;
    typedef T vT __attribute__((ext_vector_type(VL)));
    if (MODE == LOWER_T) {
#pragma unroll
        for (int c = 0; c < SB; ++c) r[c] = t[c][lane];
    } else {
#pragma unroll
        for (int c = 0; c < SB; c += VL) {
            const vT x = *reinterpret_cast<const vT *>(&t[lane][c]);
#pragma unroll
            for (int q = 0; q < VL; ++q) r[c + q] = x[q];
        }
    }
}

// With more right-hand sides than waves the update is a product of a workgroup's
// 64 rows of M, the step's 128 columns and up to 16 vectors: matrix cores, one
// 16 x 16 tile per wave.  With fewer it is a dot product per row and vector.
constexpr int RDOT = 4;

// One right-hand side of a sub-block, a column at a time: each entry divided by
// its diagonal and subtracted only from the entries after it.
template <class T, int MODE>
__device__ __forceinline__ T sweep_plain(const T (*t)[SB + TP<T>], T x, T dl, int lane) {
#pragma unroll 1
    for (int cc = 0; cc < SB; ++cc) {
        const int c = forward<MODE>() ? cc : SB - 1 - cc;
        if (MODE != LOWER_UNIT && lane == c) x = x / dl;
        const T xc = lane_get(x, c), m = MODE == LOWER_T ? t[c][lane] : t[lane][c];
        if (forward<MODE>() ? lane > c : lane < c) x = x - m * xc;
    }
    return x;
}

// The exponent of v, with |v| in [2^(e-1), 2^e); 0 for zero, infinities and NaN.
__device__ __forceinline__ int exponent(double v) { return __builtin_amdgcn_frexp_exp(v); }
__device__ __forceinline__ int exponent(float v) { return __builtin_amdgcn_frexp_expf(v); }

// Exponents below which the scaled sweep may lose bits.  A step of it is one fused
// multiply-add, exact but for its rounding, so what counts is that the quotients
// m / d are normal (NORMAL) and that no entry is so small that 64 roundings to a
// multiple of the smallest subnormal number show in it (LOW): neither the entries
// that are not zero, nor the products whose sum could have come out as zero.
// ENTRY, SOLVED and RHS are bounds on the three kinds of exponent that together
// imply both.  (They cost 1 % of a solve of order 4096, 541 to 546 us.)
template <class T> struct Range;
template <> struct Range<double> {
    static constexpr int NORMAL = -1021, LOW = -1009, ENTRY = -500, SOLVED = -500, RHS = -1000;
};
template <> struct Range<float> {
    static constexpr int NORMAL = -125, LOW = -117, ENTRY = -45, SOLVED = -70, RHS = -100;
};
// Whether the scaled sweep of a sub-block (x to y) can have lost bits; uniform.
template <class T, int MODE>
__device__ __forceinline__ bool sweep_lossy(const T (*t)[SB + TP<T>], T x, T dl, T y, int lane) {
    using R = Range<T>;
    const int ed = exponent(dl);
    int q = 0;  // the smallest quotient's exponent
#pragma unroll 8
    for (int c = 0; c < SB; ++c) {
        const T m = MODE == LOWER_T ? t[c][lane] : t[lane][c];
        q = min(q, m != T(0) ? exponent(m) - ed : 0);
    }
    q = wave_min_i32(q);
    const int s = wave_min_i32(exponent(y));
    return q < R::NORMAL || s < R::LOW || q + s < R::LOW || __any(x != T(0) && exponent(x) - ed < R::LOW);
}

// NR: right-hand sides per wave (wave w sweeps w, w + 4, ...).
template <class T, int MODE, int NR>
__global__ __launch_bounds__(256) void k_trsv_step(const T *__restrict__ M, long lda, int n, int q0,
                                                   int nq, int nrhs, T *__restrict__ W, long ldw,
                                                   T *__restrict__ X, long ldx, int u0, int u1,
                                                   int vec) {
    // tiles: [0] diagonal of sub-block 0, [1] diagonal of sub-block 1,
    // [2] the off-diagonal tile inside the stored triangle
    __shared__ __attribute__((aligned(16))) T tl[3][SB][SB + TP<T>];
    __shared__ __attribute__((aligned(16))) T xs[TMAXR][TSB * SB + TP<T>];
    __shared__ int s_low[4];  // the smallest exponent in each wave's part of the diagonal tiles
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int s0 = q0 * SB, s1 = min(n, (q0 + nq) * SB), S = s1 - s0;
    const int bs0 = min(SB, S), bs1 = S - bs0;  // rows of sub-blocks 0 and 1
    constexpr bool fwd = forward<MODE>();

    // ---- every read that does not depend on the super-block's solution is
    // issued first, so a launch waits for memory once, not once per phase:
    // the update slice and, for the first right-hand sides, its rows of W;
    // the three tiles; this wave's right-hand sides on the super-block.
    constexpr int NIT = RPW / 16, NC = TSB * SB / 16;  // row forms
    constexpr int CW = TSB * SB / 4;                   // transposed form
    constexpr bool PRODUCT = NR > 1;
    constexpr int VL = TVL<T>;
    const int ls = lane & 15, grp = lane >> 4;
    const int rbase = u0 + (int)blockIdx.x * RPW + wave * (RPW / 4) + grp;
    const int jt = u0 + (int)blockIdx.x * CPW + lane;
    // product form: the wave's 16 rows (row ls of them per lane), the lane's
    // columns 4 VL u + VL grp + e, and the W entries of its accumulator
    const int jp = u0 + (int)blockIdx.x * RPW + wave * 16;
    // No test per load: rows past u1 read row u1 - 1 (their sums are not stored), and
    // with a block of fewer than 128 columns those past it read its last column and
    // count as zero.  (Tested one by one they were waited for one by one: the last
    // workgroup of a launch, if its rows are not 64, then took 13 us where the others
    // took 7.)
    const bool rows = u1 > u0, whole = S == TSB * SB;
    const auto row_of = [&](int j) __attribute__((always_inline)) { return (long)min(j, u1 - 1); };
    T mv[PRODUCT ? CW : MODE == LOWER_T ? CW : NIT * NC];
    T wpre[PRODUCT ? 1 : RDOT][PRODUCT ? 4 : MODE == LOWER_T ? 1 : NIT];
    if constexpr (PRODUCT) {
        typedef T vT __attribute__((ext_vector_type(VL)));
        const long j = row_of(jp + ls);
        const T *const mrow = MODE == LOWER_T ? M + (long)s0 * lda + j : M + j * lda + s0;
        if (rows && whole && (vec || MODE == LOWER_T)) {
            const T *const p = MODE == LOWER_T ? mrow + (long)(grp * VL) * lda : mrow + grp * VL;
#pragma unroll
            for (int u = 0; u < CW / VL; ++u) {
                if constexpr (MODE == LOWER_T) {
#pragma unroll
                    for (int e = 0; e < VL; ++e) mv[u * VL + e] = p[(4 * u * VL + e) * lda];
                } else {
                    const vT x = *reinterpret_cast<const vT *>(p + 4 * u * VL);
#pragma unroll
                    for (int e = 0; e < VL; ++e) mv[u * VL + e] = x[e];
                }
            }
        } else if (rows && whole) {
#pragma unroll
            for (int i = 0; i < CW; ++i) mv[i] = mrow[(4 * (i / VL) + grp) * VL + i % VL];
        } else if (rows) {
#pragma unroll
            for (int i = 0; i < CW; ++i) {
                const int c = (4 * (i / VL) + grp) * VL + i % VL;
                const T v = mrow[MODE == LOWER_T ? (long)min(c, S - 1) * lda : (long)min(c, S - 1)];
                mv[i] = c < S ? v : T(0);
            }
        }
        if (rows) {  // (lanes past nrhs: the last vector's, not stored)
#pragma unroll
            for (int q = 0; q < 4; ++q) wpre[0][q] = W[(long)min(ls, nrhs - 1) * ldw + row_of(jp + Mfma<T>::row(grp, q))];
        }
    } else if constexpr (MODE == LOWER_T) {
        if (rows) {
            const T *const p = M + (long)(s0 + wave * CW) * lda + row_of(jt);
            if (whole) {
#pragma unroll
                for (int q = 0; q < CW; ++q) mv[q] = p[q * lda];
            } else {
#pragma unroll
                for (int q = 0; q < CW; ++q) {
                    const int c = wave * CW + q;
                    const T v = p[(long)(min(c, S - 1) - wave * CW) * lda];
                    mv[q] = c < S ? v : T(0);
                }
            }
            if (wave == 0) {
#pragma unroll
                for (int r = 0; r < RDOT; ++r) {
                    if (r >= nrhs) break;
                    wpre[r][0] = W[(long)r * ldw + row_of(jt)];
                }
            }
        }
    } else if (rows) {
        const T *p[NIT];
#pragma unroll
        for (int it = 0; it < NIT; ++it) p[it] = M + row_of(rbase + it * 4) * lda + s0;
        if (whole) {
#pragma unroll
            for (int it = 0; it < NIT; ++it)
#pragma unroll
                for (int k = 0; k < NC; ++k) mv[it * NC + k] = p[it][ls + 16 * k];
        } else {
#pragma unroll
            for (int it = 0; it < NIT; ++it)
#pragma unroll
                for (int k = 0; k < NC; ++k) {
                    const int c = ls + 16 * k;
                    const T v = p[it][min(c, S - 1)];
                    mv[it * NC + k] = c < S ? v : T(0);
                }
        }
#pragma unroll
        for (int r = 0; r < RDOT; ++r) {
            if (r >= nrhs) break;
#pragma unroll
            for (int it = 0; it < NIT; ++it) wpre[r][it] = W[(long)r * ldw + row_of(rbase + it * 4)];
        }
    }
    {
        T v0[TPER], v1[TPER], v2[TPER];
        const bool vf0 = vec && bs0 == SB, vf1 = vec && bs1 == SB;  // full tiles
        tile_load<T, MODE>(v0, M, lda, s0, s0, bs0, bs0, true, vec);
        if (nq > 1) {
            tile_load<T, MODE>(v1, M, lda, s0 + SB, s0 + SB, bs1, bs1, true, vec);
            if (stored_upper<MODE>())
                tile_load<T, MODE>(v2, M, lda, s0, s0 + SB, bs0, bs1, false, vec);
            else
                tile_load<T, MODE>(v2, M, lda, s0 + SB, s0, bs1, bs0, false, vec);
        }
        // this wave's right-hand sides on the two sub-blocks, and the diagonal
        T xw[2][NR], dg[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const bool in = lane < (q == 0 ? bs0 : bs1);
            const long row = s0 + q * SB + lane;
#pragma unroll
            for (int k = 0; k < NR; ++k)
                xw[q][k] = in && wave + 4 * k < nrhs ? W[(long)(wave + 4 * k) * ldw + row] : T(0);
            dg[q] = MODE != LOWER_UNIT && in && wave < nrhs ? M[row * lda + row] : T(1);
        }
        tile_store(tl[0], v0, vf0);
        if (nq > 1) {
            tile_store(tl[1], v1, vf1);
            tile_store(tl[2], v2, vf0 && vf1);
        }
        if constexpr (MODE != LOWER_UNIT) {
            int e = 0;
#pragma unroll
            for (int q = 0; q < TPER; ++q) e = min(e, exponent(v0[q]));
            if (nq > 1) {
#pragma unroll
                for (int q = 0; q < TPER; ++q) e = min(e, exponent(v1[q]));
            }
            e = wave_min_i32(e);
            if (lane == 0) s_low[wave] = e;
        }
        __syncthreads();

        // ---- 1. the super-block, redundantly in every workgroup.  The loops run
        // all 64 columns: the staged tiles are zero outside the block and x is
        // zero on lanes beyond it, so the columns past it subtract exact zeros.
        if (wave < nrhs) {
            const int low = MODE != LOWER_UNIT ? min(min(s_low[0], s_low[1]), min(s_low[2], s_low[3])) : 0;
            T sol[2][NR];
#pragma unroll
            for (int k = 0; k < NR; ++k) sol[0][k] = sol[1][k] = T(0);
#pragma unroll
            for (int qi = 0; qi < 2; ++qi) {
                if (qi >= nq) break;
                // the sub-block solved now; with one sub-block it is block 0
                const bool second = fwd ? qi == 1 : qi == 0 && nq > 1;
                T x[NR];
#pragma unroll
                for (int k = 0; k < NR; ++k) x[k] = second ? xw[1][k] : xw[0][k];
                const T dl = second ? dg[1] : dg[0];
                if (qi == 1) {  // contribution of the sub-block solved first
                    T m[SB], sum[NR];
                    tile_row<T, MODE>(tl[2], lane, m);
#pragma unroll
                    for (int k = 0; k < NR; ++k) sum[k] = T(0);
#pragma unroll
                    for (int c = 0; c < SB; ++c)
#pragma unroll
                        for (int k = 0; k < NR; ++k) sum[k] = fma(m[c], lane_get(sol[0][k], c), sum[k]);
#pragma unroll
                    for (int k = 0; k < NR; ++k) x[k] -= sum[k];
                }
                const T(*t)[SB + TP<T>] = second ? tl[1] : tl[0];
                T m[SB], y[NR];
                tile_row<T, MODE>(t, lane, m);
                if constexpr (MODE != LOWER_UNIT) {
                    const T rd = T(1) / dl;
#pragma unroll
                    for (int c = 0; c < SB; ++c) m[c] = scaled(m[c], dl, rd);
#pragma unroll
                    for (int k = 0; k < NR; ++k) y[k] = scaled(x[k], dl, rd);
                } else {
#pragma unroll
                    for (int k = 0; k < NR; ++k) y[k] = x[k];
                }
#pragma unroll
                for (int cc = 0; cc < SB; ++cc) {
                    const int c = fwd ? cc : SB - 1 - cc;
#pragma unroll
                    for (int k = 0; k < NR; ++k) y[k] = fma(-m[c], lane_get(y[k], c), y[k]);
                }
                // one test for all of them: a branch costs as much as 30 instructions
                const auto wild = [](T v) __attribute__((always_inline)) {
                    return !(fabs(v) < std::numeric_limits<T>::infinity());
                };
                bool odd = false;
#pragma unroll
                for (int k = 0; k < NR; ++k) {
                    odd |= wild(y[k]);
                    if constexpr (MODE != LOWER_UNIT) {
                        odd |= exponent(y[k]) < Range<T>::SOLVED;
                        odd |= exponent(x[k]) - exponent(dl) < Range<T>::RHS;
                    }
                }
                if constexpr (MODE != LOWER_UNIT) odd |= low - exponent(dl) < Range<T>::ENTRY;
                if (__any(odd)) {
#pragma unroll
                    for (int k = 0; k < NR; ++k)
                        if (__any(wild(y[k])) ||
                            (MODE != LOWER_UNIT && sweep_lossy<T, MODE>(t, x[k], dl, y[k], lane)))
                            y[k] = sweep_plain<T, MODE>(t, x[k], dl, lane);
                }
#pragma unroll
                for (int k = 0; k < NR; ++k) {
                    if (lane >= (second ? bs1 : bs0)) y[k] = T(0);
                    sol[qi][k] = y[k];
                }
            }
#pragma unroll
            for (int k = 0; k < NR; ++k) {
                const int r = wave + 4 * k;
                const bool swap = !fwd && nq > 1;  // block 1 was solved first
                if (r < nrhs) {
                    xs[r][lane] = swap ? sol[1][k] : sol[0][k];
                    xs[r][SB + lane] = swap ? sol[0][k] : sol[1][k];
                }
            }
        }
    }
    __syncthreads();
    if (blockIdx.x == 0)
        for (int r = wave; r < nrhs; r += 4)
            for (int c = lane; c < S; c += 64) X[(long)r * ldx + s0 + c] = xs[r][c];

    // ---- 2. remove the solved rows from this workgroup's share of [u0, u1)
    if (!rows) return;
    if constexpr (PRODUCT) {
        // four sums of 32 products each: one of 128 gave a solution of order 4096
        // 1.5 times the backward error
        typename Mfma<T>::acc part[4] = {};
#pragma unroll
        for (int u = 0; u < CW / VL; ++u)
#pragma unroll
            for (int e = 0; e < VL; ++e) {
                const int i = u * VL + e;
                part[i & 3] = Mfma<T>::op(mv[i], xs[ls][(4 * u + grp) * VL + e], part[i & 3]);
            }
        const typename Mfma<T>::acc acc = (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int jw = jp + Mfma<T>::row(grp, q);
            if (jw < u1 && ls < nrhs) W[(long)ls * ldw + jw] = wpre[0][q] - acc[q];
        }
    } else if constexpr (MODE == LOWER_T) {
        // W[r][j] -= sum_c L[s0 + c][j] * x[c]: a workgroup owns 64 entries j
        // (one per lane: coalesced rows of L), wave w sums c in [32w, 32w + 32)
        const bool act = jt < u1;
        // partial sums meet in LDS (the staged tiles are no longer read)
        T(*red)[RDOT][SB] = reinterpret_cast<T(*)[RDOT][SB]>(&tl[0][0][0]);
#pragma unroll
        for (int r = 0; r < RDOT; ++r) {
            if (r >= nrhs) break;
            T a = T(0);
#pragma unroll
            for (int q = 0; q < CW; ++q) a += mv[q] * xs[r][wave * CW + q];
            red[wave][r][lane] = a;
        }
        __syncthreads();
        if (wave == 0 && act) {
#pragma unroll
            for (int r = 0; r < RDOT; ++r) {
                if (r >= nrhs) break;
                const T a = (red[0][r][lane] + red[1][r][lane]) + (red[2][r][lane] + red[3][r][lane]);
                W[(long)r * ldw + jt] = wpre[r][0] - a;
            }
        }
    } else {
        // W[r][j] -= sum_c M[j][s0 + c] * x[c]; 16 lanes per row, 4 rows per
        // wave at a time, lane ls holds columns ls, ls + 16, ... (coalesced)
#pragma unroll
        for (int r = 0; r < RDOT; ++r) {
            if (r >= nrhs) break;
            T v[NIT];
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
                T a = T(0);
#pragma unroll
                for (int k = 0; k < NC; ++k) a += mv[it * NC + k] * xs[r][ls + 16 * k];
                v[it] = row16_sum(a);  // the 16 lanes of a row are one DPP row
            }
            if (ls == 0) {
#pragma unroll
                for (int it = 0; it < NIT; ++it) {
                    const int j = rbase + it * 4;
                    if (j < u1) W[(long)r * ldw + j] = wpre[r][it] - v[it];
                }
            }
        }
    }
}

template <class T, int MODE>
static int trsv_run(hipStream_t s, size_t n, const T *m, size_t lda, size_t nrhs, T *w, size_t ldw,
                    T *x, size_t ldx) {
    if (n == 0 || nrhs == 0) return RLG_OK;
    if (w == x) {
        set_error("triangular solve: residual and output buffers must differ");
        return RLG_E_INVALID_ARG;
    }
    constexpr bool fwd = MODE == LOWER_UNIT || MODE == LOWER;
    // 16-byte tile loads when rows of the triangle start 16-byte aligned
    const bool vec = lda % TVL<T> == 0 && (reinterpret_cast<uintptr_t>(m) & 15) == 0;
    const size_t nb = (n + SB - 1) / SB;
    const size_t steps = (nb + TSB - 1) / TSB;
    for (size_t r0 = 0; r0 < nrhs; r0 += TMAXR) {
        const size_t nr = nrhs - r0 < (size_t)TMAXR ? nrhs - r0 : TMAXR;
        for (size_t k = 0; k < steps; ++k) {
            size_t q0, nq;
            if (fwd) {
                q0 = k * TSB;
                nq = nb - q0 < (size_t)TSB ? nb - q0 : TSB;
            } else {
                const size_t qe = nb - k * TSB;
                q0 = qe > (size_t)TSB ? qe - TSB : 0;
                nq = qe - q0;
            }
            const size_t s0 = q0 * SB, s1 = (q0 + nq) * SB < n ? (q0 + nq) * SB : n;
            const size_t u0 = fwd ? s1 : 0, u1 = fwd ? n : s0;
            const size_t per = MODE == LOWER_T ? CPW : RPW;
            const unsigned grid = u1 > u0 ? ceil_div(u1 - u0, per) : 1u;
            // algorithmic bytes: the super-block triangle, the update slice,
            // the right-hand-side rows read and written
            const double bytes =
                sizeof(T) * ((double)(s1 - s0) * (s1 - s0 + 1) / 2 + (double)(u1 - u0) * (s1 - s0) +
                             (double)nr * (2.0 * (u1 - u0) + 2.0 * (s1 - s0)));
            RLG_PROF_W("trsv", s, bytes);
            auto go = [&](auto nr_wave) {
                hipLaunchKernelGGL((k_trsv_step<T, MODE, decltype(nr_wave)::value>), dim3(grid), dim3(256), 0,
                                   s, m, (long)lda, (int)n, (int)q0, (int)nq, (int)nr, w + r0 * ldw, (long)ldw,
                                   x + r0 * ldx, (long)ldx, (int)u0, (int)u1, vec ? 1 : 0);
            };
            // four waves: as few right-hand sides per wave as hold them all
            if (nr <= (size_t)RDOT) go(std::integral_constant<int, 1>{});
            else if (nr <= 8) go(std::integral_constant<int, 2>{});
            else go(std::integral_constant<int, 4>{});
            RLG_LAUNCHED();
        }
    }
    return RLG_OK;
}

template <class T>
int trsv_lower(hipStream_t s, size_t n, const T *l, size_t lda, bool unit, size_t nrhs, T *in,
               size_t ldi, T *out, size_t ldo) {
    return unit ? trsv_run<T, LOWER_UNIT>(s, n, l, lda, nrhs, in, ldi, out, ldo)
                : trsv_run<T, LOWER>(s, n, l, lda, nrhs, in, ldi, out, ldo);
}

template <class T>
int trsv_upper(hipStream_t s, size_t n, const T *u, size_t lda, size_t nrhs, T *in, size_t ldi,
               T *out, size_t ldo) {
    return trsv_run<T, UPPER>(s, n, u, lda, nrhs, in, ldi, out, ldo);
}

template <class T>
int trsv_lower_t(hipStream_t s, size_t n, const T *l, size_t lda, size_t nrhs, T *in, size_t ldi,
                 T *out, size_t ldo) {
    return trsv_run<T, LOWER_T>(s, n, l, lda, nrhs, in, ldi, out, ldo);
}

// The singularity test of back_substitution and forward_substitution
// (src/matrix/mod.rs:331-335, 375-378): a diagonal entry below epsilon in
// magnitude.  Every flagged lane stores the same value with a vector store.
template <class T>
__global__ void k_diag_tiny(const T *__restrict__ M, long lda, long n, T eps, uint32_t *flag) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && std::fabs(M[i * lda + i]) < eps) *flag = 1u;
}

template <class T>
int diag_tiny(hipStream_t s, size_t n, const T *m, size_t lda, T eps, uint32_t *flag) {
    if (n == 0) return RLG_OK;
    hipLaunchKernelGGL(k_diag_tiny<T>, dim3(ceil_div(n, 256)), dim3(256), 0, s, m, (long)lda,
                       (long)n, eps, flag);
    RLG_LAUNCHED();
    return RLG_OK;
}
template int diag_tiny<double>(hipStream_t, size_t, const double *, size_t, double, uint32_t *);
template int diag_tiny<float>(hipStream_t, size_t, const float *, size_t, float, uint32_t *);

#define RLG_TRSV_INST(T)                                                                           \
    template int trsv_lower<T>(hipStream_t, size_t, const T *, size_t, bool, size_t, T *, size_t, \
                               T *, size_t);                                                       \
    template int trsv_upper<T>(hipStream_t, size_t, const T *, size_t, size_t, T *, size_t, T *,   \
                               size_t);                                                            \
    template int trsv_lower_t<T>(hipStream_t, size_t, const T *, size_t, size_t, T *, size_t, T *, \
                                 size_t);
RLG_TRSV_INST(double)
RLG_TRSV_INST(float)

}  // namespace rlg
