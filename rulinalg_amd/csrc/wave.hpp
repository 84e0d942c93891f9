// Wave-level helpers for gfx950 (wave64): lane broadcasts and reductions over
// the wave built from DPP moves, which cost a few cycles each, where a
// shuffle through the LDS crossbar (ds_bpermute) costs about a hundred.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>
#include <utility>

namespace rlg {

// Calls f(std::integral_constant<int, I>) for I = 0 .. N-1 in order, so a
// loop body sees its index as a compile-time constant and registers indexed
// by it stay registers.
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F &f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}


// Value of x in lane `l` (uniform result).
__device__ __forceinline__ int lane_get(int x, int l) { return __builtin_amdgcn_readlane(x, l); }
__device__ __forceinline__ float lane_get(float x, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
__device__ __forceinline__ double lane_get(double x, int l) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// DPP lane permutations within rows of 16 lanes.
constexpr int DPP_XOR1 = 0xB1;         // quad_perm [1, 0, 3, 2]
constexpr int DPP_XOR2 = 0x4E;         // quad_perm [2, 3, 0, 1]
constexpr int DPP_HALF_MIRROR = 0x141; // lane i <-> 7 - i within each 8
constexpr int DPP_MIRROR = 0x140;      // lane i <-> 15 - i within each 16

template <int N> constexpr int DPP_SHR = 0x110 + N;  // lane i <- lane i - N within each 16
constexpr int DPP_BCAST15 = 0x142;     // a row's lane 15 -> the next row
constexpr int DPP_BCAST31 = 0x143;     // lane 31 -> lanes 32..63

template <int CTRL> __device__ __forceinline__ int dpp(int x) {
    return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false);
}
template <int CTRL> __device__ __forceinline__ float dpp(float x) {
    return __int_as_float(dpp<CTRL>(__float_as_int(x)));
}
template <int CTRL> __device__ __forceinline__ double dpp(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = dpp<CTRL>((int)b), hi = dpp<CTRL>((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// The value again, unknown to the compiler: addresses made from it are formed
// where they are used, not ahead of a loop and kept in scratch memory.
__device__ __forceinline__ int opaque(int v) {
#ifdef __AMDGCN__
    asm volatile("" : "+v"(v));
#endif
    return v;
}

#ifdef __AMDGCN__
// The value, known to be the same in every lane.
__device__ __forceinline__ unsigned long long uniform(unsigned long long v) {
    return ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
           (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}
// b where this lane's bit of the (uniform) mask is clear, else a.
template <class V> __device__ __forceinline__ V bit_of(unsigned long long mask, V a, V b) {
    return __builtin_amdgcn_inverse_ballot_w64(mask) ? a : b;
}
#endif

// Maximum of a 32-bit key over the wave (uniform result): two quad swaps
// and two row mirrors, then the four rows' maxima from lanes 0, 16, 32, 48.
__device__ __forceinline__ unsigned lane_get(unsigned x, int l) {
    return (unsigned)__builtin_amdgcn_readlane((int)x, l);
}
// max(x, x of the lane CTRL names): bound control with a zero fill lets the
// compiler fuse the move into the maximum.
template <int CTRL> __device__ __forceinline__ unsigned dpp_max(unsigned x) {
    const unsigned y = (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, true);
    return x > y ? x : y;
}
__device__ __forceinline__ unsigned wave_max_u32(unsigned k) {
    auto mx = [](unsigned a, unsigned b) { return a > b ? a : b; };
    k = dpp_max<DPP_XOR1>(k);
    k = dpp_max<DPP_XOR2>(k);
    k = dpp_max<DPP_HALF_MIRROR>(k);
    k = dpp_max<DPP_MIRROR>(k);
    return mx(mx(lane_get(k, 0), lane_get(k, 16)), mx(lane_get(k, 32), lane_get(k, 48)));
}

// Sum over each row of 16 lanes, in every lane of the row: four rotations
// within the row (row_ror 8, 4, 2, 1), each a DPP move.
template <int N> constexpr int DPP_ROR = 0x120 + N;
template <class T> __device__ __forceinline__ T row16_sum(T a) {
    a += dpp<DPP_ROR<8>>(a);
    a += dpp<DPP_ROR<4>>(a);
    a += dpp<DPP_ROR<2>>(a);
    a += dpp<DPP_ROR<1>>(a);
    return a;
}

// Minimum of an int over the wave (uniform result), the same pattern.
__device__ __forceinline__ int wave_min_i32(int k) {
    k = min(k, dpp<DPP_XOR1>(k));
    k = min(k, dpp<DPP_XOR2>(k));
    k = min(k, dpp<DPP_HALF_MIRROR>(k));
    k = min(k, dpp<DPP_MIRROR>(k));
    return min(min(lane_get(k, 0), lane_get(k, 16)), min(lane_get(k, 32), lane_get(k, 48)));
}

// ---------------------------------------------------------------- pivot search

// Candidate order: larger magnitude first; equal magnitudes go to the lower
// row index.  That is the reference's scan from the diagonal down, which takes a row
// only if it is larger than the best before it: a NaN is never taken, and one on the
// diagonal never given up.

// The high word of a magnitude plus one (a non-negative float orders like its
// bits); a NaN ranks like zero, but in the diagonal's row by its bits, which are at
// least infinity's (the tie that leaves goes to the lower row, the diagonal's).
__device__ __forceinline__ unsigned rank_hi(float v, bool diagonal) {
    return (int)(v == v) | (int)diagonal ? __float_as_uint(v) + 1 : 1u;
}
__device__ __forceinline__ unsigned rank_hi(double v, bool diagonal) {
    return (int)(v == v) | (int)diagonal ? (unsigned)((unsigned long long)__double_as_longlong(v) >> 32) + 1 : 1u;
}
__device__ __forceinline__ unsigned rank_lo(float) { return 0u; }
__device__ __forceinline__ unsigned rank_lo(double v) {
    return (v == v) ? (unsigned)(unsigned long long)__double_as_longlong(v) : 0u;
}

// The lane that holds the wave's first maximum (largest |value|, ties to the
// smallest row index i), or -1 if no lane has a candidate;
// uniform.  A lane without one passes hi = 0, else the ranks of its value.  The
// high words settle it but for near-ties: one 32-bit maximum over the wave, a
// fused DPP instruction per step, where a 64-bit one takes a compare and two
// selects (610 against about 380 cycles).  Then the low words, then the indices.
__device__ __forceinline__ int first_max_lane(unsigned hi, unsigned lo, int i) {
    const unsigned mh = wave_max_u32(hi);
    if (mh == 0) return -1;
    const unsigned long long tied = __ballot(hi == mh);
    if (__popcll(tied) == 1) return __ffsll((long long)tied) - 1;
    const unsigned ml = wave_max_u32(hi == mh ? lo : 0u);
    const int ii = hi == mh && lo == ml ? i : INT_MAX;
    const int mi = wave_min_i32(ii);
    return __ffsll((long long)__ballot(ii == mi)) - 1;
}

}  // namespace rlg
