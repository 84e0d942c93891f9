// Right-looking blocked LU with partial pivoting (PartialPivLu::decompose,
// src/matrix/decomposition/lu.rs:163-194) and its solve (lu.rs:231-244).
//
// Blocking: outer blocks of ONB = 512 columns drive the trailing Schur
// update as one MFMA GEMM of depth 512 (faster than 256 at order 16384 in
// both FP64 and FP32: less C traffic per flop); inside an outer block, inner panels
// of PNB = 64 columns are factored by a kernel launched cooperatively
// (hipLaunchCooperativeKernel: all of its workgroups resident together) and
// applied to the rest of the outer block by a 64-row triangular solve and a
// depth-64 GEMM.
//
// The panel kernel keeps the whole (n - k) x 64 panel resident in LDS,
// spread over G workgroups of PanelRows rows each, and factors it 16 columns at a
// time with a row's 16 entries in its thread's registers (see k_lu_panel).
// With more than one workgroup every column costs one exchange: each publishes
// its pivot candidate (|value|, row, and the row's 16 entries) as tagged words;
// every workgroup reads the G candidates and reduces them to the same winner.
// The pivot rule is the reference's: the first row of maximal magnitude at or
// below the diagonal (strict `>` scan, lu.rs:170-178).  An order of at most 64
// is factored bit-identically to the reference: there the multiplier is a
// division and the update a separately rounded multiply and subtract
// (lu.rs:603-616).
#include <climits>
#include <type_traits>

#include "kernels.hpp"
#include "mfma.hpp"
#include "recip.hpp"
#include "wave.hpp"

namespace rlg {

constexpr int PNB = 64;    // inner panel width
constexpr int SPW = 16;    // columns held in registers at a time
// Panel rows per workgroup (LDS-resident), one per thread: 256 in FP64
// (154,592 bytes of LDS, one workgroup per CU, so every workgroup of a panel is
// resident at once) and 512 in FP32 (151,648 bytes).
template <class T> struct PanelRows { static constexpr int value = 256; };
template <> struct PanelRows<float> { static constexpr int value = 512; };
constexpr int ONB = 512;   // outer block: depth of the trailing GEMM
constexpr int SWB = 256;   // swaps per k_laswp launch (its workgroup size)
// At most this many workgroups per panel: one per CU of the device and never
// more than the exchange area holds.
constexpr int GMAX = 256;

template <class T> __device__ __forceinline__ T eps_of();
template <> __device__ __forceinline__ double eps_of<double>() { return 2.220446049250313e-16; }
template <> __device__ __forceinline__ float eps_of<float>() { return 1.1920929e-7f; }

// Exchange words of the panel workgroups.  A 64-bit word carries 32 bits of
// payload in its low half and, in its high half, the tag of the column it
// belongs to: global column + 1, 0 = never written in this factorization.
// Words are written and read with agent-scope atomics, and a reader polls
// until every word it needs carries the current tag, so a value is never
// used before it is complete and no counter, fence or barrier is involved.
// A candidate slot holds a header, the low word of |value| (read only to settle
// a tie) and the row's entries in the 16 columns at hand; a pivot-row slot holds
// a pivot row from those columns on.  A value takes one word in FP32 and two
// (low, high half) in FP64.  The header is one word, so that a poll is one
// load: the high word of |value| (rank_hi; 0: no candidate), the row in 17 bits
// and the low 15 bits of the tag, which suffice since a slot's last content is
// two columns old.
typedef unsigned long long xword;
constexpr int XHDR = 2;  // header and the low word of |value|
__device__ __forceinline__ xword xhdr(unsigned hi, int row, unsigned tag) {
    return ((xword)hi << 32) | ((unsigned)row << 15) | (tag & 0x7fffu);
}
template <class T> struct XSlot {
    static constexpr int VW = sizeof(T) / 4;                      // words per value
    static constexpr int words = (XHDR + SPW * VW + 15) & ~15;    // 128-byte multiple
    static constexpr int parity = GMAX * words;                   // candidates of one column parity
    static constexpr int rows = SPW * PNB * VW;                   // pivot rows of one 16-column parity
};

// Workspace layout (bytes): exchange slots, inverses of the unit-lower
// diagonal blocks of the current outer block, timeout flag.
struct LuWork {
    xword *xch;        // candidates [2][GMAX][words], then pivot rows [2][SPW][PNB]
    void *linv;        // [ONB / PNB][PNB][PNB] T
    int *timeout;      // exchange timeout flag
};

static size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }
static size_t xch_words(size_t elem) {
    return 2 * (size_t)(elem == 8 ? XSlot<double>::parity + XSlot<double>::rows
                                  : XSlot<float>::parity + XSlot<float>::rows);
}

size_t lu_work_bytes(size_t n, size_t elem) {
    (void)n;
    return align_up(xch_words(elem) * sizeof(xword)) + align_up((size_t)ONB * PNB * elem) +
           align_up(4);
}

static LuWork carve(void *work, size_t n, size_t elem) {
    (void)n;
    char *p = static_cast<char *>(work);
    LuWork w;
    w.xch = reinterpret_cast<xword *>(p); p += align_up(xch_words(elem) * sizeof(xword));
    w.linv = p; p += align_up((size_t)ONB * PNB * elem);
    w.timeout = reinterpret_cast<int *>(p);
    return w;
}

int *lu_timeout_flag(void *work, size_t n, size_t elem) { return carve(work, n, elem).timeout; }

void perm_from_ipiv(size_t n, const int64_t *ipiv, int64_t *raw) {
    for (size_t i = 0; i < n; ++i) raw[i] = (int64_t)i;
    for (size_t k = 0; k < n; ++k) {
        const size_t p = (size_t)ipiv[k];
        if (p != k) { int64_t t = raw[k]; raw[k] = raw[p]; raw[p] = t; }
    }
}

// ---------------------------------------------------------------- panel

__device__ __forceinline__ unsigned xtag(xword w) { return (unsigned)(w >> 32); }
__device__ __forceinline__ void xput(xword *p, unsigned tag, unsigned v) {
    __hip_atomic_store(p, ((xword)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ xword xget(const xword *p) {
    return __hip_atomic_load(const_cast<xword *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void xput_val(xword *p, unsigned tag, float v) {
    xput(p, tag, __float_as_uint(v));
}
__device__ __forceinline__ void xput_val(xword *p, unsigned tag, double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    xput(p, tag, (unsigned)b);
    xput(p + 1, tag, (unsigned)(b >> 32));
}
// The value at p; ok = every word of it carries `tag`.
template <class T> __device__ __forceinline__ T xget_val(const xword *p, unsigned tag, bool &ok);
template <> __device__ __forceinline__ float xget_val<float>(const xword *p, unsigned tag, bool &ok) {
    const xword a = xget(p);
    ok = xtag(a) == tag;
    return __uint_as_float((unsigned)a);
}
template <> __device__ __forceinline__ double xget_val<double>(const xword *p, unsigned tag, bool &ok) {
    const xword a = xget(p), b = xget(p + 1);
    ok = xtag(a) == tag && xtag(b) == tag;
    return __longlong_as_double((long long)(((b & 0xffffffffull) << 32) | (a & 0xffffffffull)));
}

constexpr int XPOLLS = 6;  // header loads in flight, and their spacing in sleeps of 64 cycles
constexpr int XPOLL_SLEEP = 6, XPOLL_GAP = 2;
// Up to this many workgroups (16,384 rows in FP64), the candidates' entries are
// read ahead, this many sleeps after the choice of the workgroup's own.  (From 8
// to 16 sleeps, and from 3 to 8 header loads, the time of a factorization
// differs by 1 %.)
constexpr int XROWS = 64, XROWS_SLEEP = 12;

// One round of a bounded wave-wide wait.  Returns false once the timeout
// flag is up (checked every 256 rounds) or after 2^22 rounds, when it raises
// the flag itself: an exchange that cannot complete then ends the kernel,
// and the host reports the flag, instead of hanging.  The result is uniform
// over the wave.
__device__ __forceinline__ bool xwait(unsigned &spins, int *timeout) {
    if ((++spins & 255u) == 0) {
        const int up = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(timeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (up) return false;
        if (spins >= (1u << 22)) {
            if ((threadIdx.x & 63) == 0)
                __hip_atomic_store(timeout, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
    }
    __builtin_amdgcn_s_sleep(1);
    return true;
}

// The header at h once it carries `tag` in every lane (a wave-wide wait, given
// up like xwait's).  A word takes about 1,450 cycles from one workgroup to
// another and a load's round trip is about 1,000, so several loads are kept in
// flight: polled one at a time, a word would be seen up to a round trip late.
__device__ __forceinline__ xword xpoll(const xword *h, unsigned tag, bool &live, int *timeout) {
    constexpr int N = XPOLLS;
    xword v[N];
    __builtin_amdgcn_s_sleep(XPOLL_SLEEP);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if (i) __builtin_amdgcn_s_sleep(XPOLL_GAP);
        v[i] = xget(h);
    }
    for (unsigned spins = 0;;) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (__all(((unsigned)v[i] & 0x7fffu) == (tag & 0x7fffu))) return v[i];
            v[i] = xget(h);
        }
        if (!xwait(spins, timeout)) { live = false; return 0; }
    }
}
// The payload of the word at w once it carries `tag` in every lane, bounded
// like xpoll.
__device__ __forceinline__ unsigned xlow(const xword *w, unsigned tag, bool &live, int *timeout) {
    for (unsigned spins = 0;;) {
        const xword v = xget(w);
        if (__all(xtag(v) == tag)) return (unsigned)v;
        if (!xwait(spins, timeout)) { live = false; return 0; }
    }
}

// Tile rows are padded to a 16-byte multiple: 16-byte aligned rows let a
// thread move its row with 16-byte LDS accesses, and a wave's rows then cover
// all banks.
template <class T> struct TilePad { static constexpr int value = 16 / sizeof(T); };
template <class T> constexpr int TW = PNB + TilePad<T>::value;

// Factor the panel A[k:k+m, k:k+w] (w <= PNB) in place.
//
// Workgroup g loads rows [g PRT, (g+1) PRT) of the panel into LDS, one per
// thread, and a row stays with its thread: a swap only exchanges two rows'
// positions (pos), and the rows are written to their positions at the end, when
// every workgroup has long read its own (each took part in column 0's
// exchange).  Sixteen columns at a time are held in registers.  Column j:
//   - each wave finds its first maximum over the rows at positions >= j and
//     copies that row's 16 entries to LDS; barrier; every wave picks the
//     workgroup's candidate;
//   - with other workgroups, wave 0 publishes a header (position, |value|),
//     reads all G headers and picks the same winner as every other workgroup;
//     meanwhile wave 1 publishes the candidate's entries and waves 1.. read the
//     other candidates' (at order 4,096 8 % of the factorization
//     less than fetching the winner's entries after the choice);
//     barrier; the winner's workgroup publishes the row from these columns on;
//   - rows at positions > j form their multiplier and subtract the pivot row's
//     entries right of j, in registers.
// After 16 columns the pivot rows' part right of them (from LDS, or published)
// is solved against the 16 x 16 unit-lower block and subtracted from the
// remaining rows on the matrix cores.
//
// Bound by the serial chain per column (search, barrier, exchange), not by the
// arithmetic.  Rows of 64 kept in LDS with three barriers per column and an
// update of the whole row per column took, in FP64, 122 us for a panel of 256
// rows and, on average over the factorization, 188 at order 1,531 and 209 at
// 16,384; this form takes 68, 152 to 165 (on different cards) and 189.
//
// EXACT (FP32, and FP64 orders up to 64): divisions, and separately rounded
// products and differences in the reference's order.
template <class T, bool EXACT>
__global__ __launch_bounds__(PanelRows<T>::value) void k_lu_panel(
    T *__restrict__ A, long lda, int k, int m, int w, int64_t *__restrict__ ipiv,
    int64_t *__restrict__ info, int n, xword *__restrict__ xch, int *timeout) {
    constexpr int PRT = PanelRows<T>::value;
    constexpr int NW = PRT / 64;
    using X = XSlot<T>;
    __shared__ __attribute__((aligned(16))) T tile[PRT][TW<T>];
    __shared__ __attribute__((aligned(16))) T urow[SPW][TW<T>];      // pivot rows of these columns
    __shared__ __attribute__((aligned(16))) T cand[2][NW][SPW];      // wave candidates' entries
    __shared__ __attribute__((aligned(16))) T rows_in[XROWS][SPW];   // other workgroups'
    // wave candidates: ranks of |value| (rank_hi, rank_lo; 0: none), position, thread
    __shared__ uint4 red[2][NW];
    __shared__ int4 s_win[2];     // the winner's position, workgroup, and thread here or -1
    __shared__ int s_got[XROWS];  // whether rows_in[] is complete
    __shared__ int s_piv[PNB], s_pos[PRT], s_row[SPW];

    const int G = gridDim.x, g = blockIdx.x, tid = threadIdx.x;
    const int r0 = g * PRT;
    const int rows = min(PRT, m - r0);
    const int lane = tid & 63, wave = tid >> 6;

    {   // all loads in flight before the LDS stores (64 values per thread)
        T v[PNB];
#pragma unroll
        for (int q = 0; q < PNB; ++q) {
            const int r = q * NW + wave;
            v[q] = (r < rows && lane < w) ? A[(long)(k + r0 + r) * lda + k + lane] : T(0);
        }
#pragma unroll
        for (int q = 0; q < PNB; ++q) tile[q * NW + wave][lane] = v[q];  // zero past w and m
    }
    __syncthreads();

    bool live = true;  // false once a wait of this wave has timed out
    int small = w;     // first column whose pivot is below epsilon
    int pos = tid < rows ? r0 + tid : -1;
    for (int cb = 0; cb < w; cb += SPW) {
        xword *const prows = xch + 2 * X::parity + ((cb / SPW) & 1) * X::rows;
        T x[SPW];
#pragma unroll
        for (int c = 0; c < SPW; ++c) x[c] = tile[tid][cb + c];
        if (tid < SPW) s_row[tid] = -1;
        // x[e] is the row's entry in column j + e: a column leaves the registers
        // when it is done, so one loop body serves all 16 (expanded, they would
        // be twice the instruction cache)
#pragma unroll 1
        for (int j = cb; j < min(cb + SPW, w); ++j) {
            const int c = j - cb, par = j & 1;
            const T av = fabs(x[0]);
            // (opaque: its tests' masks would be kept for the swap below, and spilled)
            const int ahead = opaque(pos - j);
            const unsigned hi = ahead >= 0 ? rank_hi(av, ahead == 0) : 0u, lo = rank_lo(av);
            const int wl = first_max_lane(hi, lo, pos);
            if (lane == max(wl, 0)) {
                red[par][wave] = uint4{wl < 0 ? 0u : hi, lo, (unsigned)pos, (unsigned)tid};
#pragma unroll
                for (int e = 0; e < SPW / 2; ++e) cand[par][wave][e] = x[e];
                if (c < SPW / 2) {  // later, the rest are past the 16 columns
#pragma unroll
                    for (int e = SPW / 2; e < SPW; ++e) cand[par][wave][e] = x[e];
                }
            }
            __syncthreads();
            const uint4 rw = red[par][lane % NW];
            unsigned top = dpp_max<DPP_XOR2>(dpp_max<DPP_XOR1>(rw.x));  // over each NW lanes
            if constexpr (NW > 4) top = dpp_max<DPP_HALF_MIRROR>(top);
            const unsigned tied = (unsigned)__ballot(rw.x == top) & ((1u << NW) - 1);
            int bw = __builtin_ctz(tied);
            if (tied & (tied - 1)) bw = max(first_max_lane(lane < NW ? rw.x : 0u, rw.y, (int)rw.z), 0);
            int p = lane_get((int)rw.z, bw), t = lane_get((int)rw.w, bw);
            const T *pr = cand[par][bw];
            if (G > 1) {
                const unsigned tag = (unsigned)(k + j + 1);
                xword *const base = xch + par * X::parity;
                xword *const slot = base + (size_t)g * X::words;
                const unsigned whi = lane_get(rw.x, bw);
                if (wave == 0) {
                    if (live && lane == 0) {
                        __hip_atomic_store(slot, xhdr(whi, whi ? p : 0, tag), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                        xput(slot + 1, tag, lane_get(rw.y, bw));
                    }
                    // every workgroup's header, 64 per round: lanes past G have none
                    unsigned bh = 0, bl = 0;
                    int i = INT_MAX, gw = g;
                    for (int q0 = 0; q0 < G && live; q0 += 64) {
                        const int q = q0 + lane;
                        const xword *h = base + (size_t)min(q, G - 1) * X::words;
                        const xword hw = xpoll(h, tag, live, timeout);
                        const unsigned qh = q < G ? (unsigned)(hw >> 32) : 0u;
                        const int qi = (int)((unsigned)hw >> 15);
                        if (G <= 64) {
                            bh = qh;
                            i = qi;
                            gw = q;
                        } else {  // a tie between rounds needs the low words now
                            const unsigned ql = xlow(h + 1, tag, live, timeout);
                            const bool take = (qh > bh) | ((qh == bh) & ((ql > bl) | ((ql == bl) & (qi < i))));
                            bh = take ? qh : bh;
                            bl = take ? ql : bl;
                            i = take ? qi : i;
                            gw = take ? q : gw;
                        }
                    }
                    const unsigned mh = wave_max_u32(bh);
                    const unsigned long long at = __ballot(bh == mh);
                    int win = __ffsll((long long)at) - 1;
                    if (__popcll(at) > 1) {
                        if (G <= 64) bl = xlow(base + (size_t)min(gw, G - 1) * X::words + 1, tag, live, timeout);
                        win = first_max_lane(bh == mh ? bh : 0u, bl, i);
                    }
                    if (live && mh) {
                        p = lane_get(i, win);
                        gw = lane_get(gw, win);
                    } else {  // no candidate anywhere cannot happen; report it
                        if (live && lane == 0)
                            __hip_atomic_store(timeout, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        live = false;
                        gw = g;  // the result is discarded: keep indices in range
                        p = j;
                        t = -1;
                    }
                    if (lane == 0) {
                        s_win[par] = int4{p, gw, gw == g ? t : -1, 0};
                        if (G > XROWS) s_got[0] = 0;
                    }
                } else {
                    if (wave == 1 && whi && lane < SPW) xput_val(slot + XHDR + lane * X::VW, tag, pr[lane]);
                    // Meanwhile the candidates' entries: the choice takes about as
                    // long as they take to arrive.
                    if (G <= XROWS) {
                        constexpr int WPR = SPW * X::VW, PW = 64 / WPR;  // words per row, rows per load
                        constexpr int LD = (XROWS + PW * (NW - 1) - 1) / (PW * (NW - 1));
                        unsigned *const rw32 = reinterpret_cast<unsigned *>(&rows_in[0][0]);
                        __builtin_amdgcn_s_sleep(XROWS_SLEEP);
                        xword v[LD];
#pragma unroll
                        for (int q = 0; q < LD; ++q) {
                            const int r = (q * (NW - 1) + wave - 1) * PW + lane / WPR;
                            v[q] = r < G ? xget(base + (size_t)r * X::words + XHDR + lane % WPR) : 0;
                        }
#pragma unroll
                        for (int q = 0; q < LD; ++q) {
                            const int r = (q * (NW - 1) + wave - 1) * PW + lane / WPR;
                            const unsigned long long good = __ballot(xtag(v[q]) == tag);
                            constexpr unsigned long long one = WPR == 64 ? ~0ull : (1ull << WPR) - 1;
                            if (r < G) {
                                rw32[r * WPR + lane % WPR] = (unsigned)v[q];
                                if (lane % WPR == 0) s_got[r] = ((good >> (lane / WPR * WPR)) & one) == one;
                            }
                        }
                    }
                }
                __syncthreads();
                const int4 sw = s_win[par];
                p = __builtin_amdgcn_readfirstlane(sw.x);
                t = __builtin_amdgcn_readfirstlane(sw.z);
                const int gw = __builtin_amdgcn_readfirstlane(sw.y);
                if (gw != g) {
                    pr = rows_in[G <= XROWS ? gw : 0];
                    if (!__builtin_amdgcn_readfirstlane(s_got[G <= XROWS ? gw : 0])) {  // not there yet
                        if (wave == 0) {
                            T pv = T(0);
                            for (unsigned spins = 0; live;) {
                                bool ok = true;
                                if (lane < SPW) pv = xget_val<T>(base + (size_t)gw * X::words + XHDR + lane * X::VW, tag, ok);
                                if (__all(ok)) break;
                                if (!xwait(spins, timeout)) live = false;
                            }
                            if (lane < SPW) rows_in[G <= XROWS ? gw : 0][lane] = pv;
                        }
                        __syncthreads();
                    }
                }
                // the winner's row from column cb on, for every workgroup's update
                if (wave == 1 && t >= 0 && cb + SPW < w && cb + lane < PNB)
                    xput_val(prows + (c * PNB + lane) * X::VW, tag,
                             lane >= c && lane < SPW ? pr[lane - c] : tile[t][cb + lane]);
            }
            const T piv = pr[0];
            if (fabs(piv) < eps_of<T>() && small == w) small = j;
            // a pivot row held here: its entries leave the registers
            if (wave == 2 && t >= 0 && lane < SPW - c) tile[t][j + lane] = pr[lane];
            if (tid == 0) s_piv[j] = p;
            if (pos == p) { pos = j; s_row[c] = tid; }
            else if (pos == j) pos = p;
            if (pos > j) {
                if constexpr (EXACT) {
#pragma clang fp contract(off)
                    const T mult = x[0] / piv;
                    tile[tid][j] = mult;
#pragma unroll
                    for (int e = 1; e < SPW; ++e) x[e - 1] = x[e] - mult * pr[e];
                } else {
                    const T mult = div_recip(x[0], piv, recip(piv));
                    tile[tid][j] = mult;
#pragma unroll
                    for (int e = 1; e <= SPW / 2; ++e) x[e - 1] = fma(-mult, pr[e], x[e]);
                    if (c < SPW / 2) {
#pragma unroll
                        for (int e = SPW / 2 + 1; e < SPW; ++e) x[e - 1] = fma(-mult, pr[e], x[e]);
                    }
                }
            }
        }
        s_pos[tid] = pos;
        if (cb + SPW >= w) break;
        __syncthreads();

        // the pivot rows from column cb on
        constexpr int PER = SPW * PNB / PRT;
        if (G == 1) {
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const int i = q * NW + wave;
                if (cb + lane < PNB) urow[i][lane] = tile[s_row[i]][cb + lane];
            }
        } else {
            T v[PER];
            for (unsigned spins = 0; live;) {
                bool ok = true;
#pragma unroll
                for (int q = 0; q < PER; ++q) {
                    const int i = q * NW + wave;
                    bool o = true;
                    v[q] = T(0);
                    if (cb + lane < PNB)
                        v[q] = xget_val<T>(prows + (i * PNB + lane) * X::VW, (unsigned)(k + cb + i + 1), o);
                    ok = ok && o;
                }
                if (__all(ok)) break;
                if (!xwait(spins, timeout)) { live = false; break; }
            }
#pragma unroll
            for (int q = 0; q < PER; ++q) urow[q * NW + wave][lane] = live ? v[q] : T(0);
        }
        __syncthreads();
        // U12 = L11^-1 A12, one column per lane
        if (wave == 0 && lane < PNB - SPW - cb) {
            T u[SPW];
#pragma unroll
            for (int i = 0; i < SPW; ++i) u[i] = urow[i][SPW + lane];
#pragma unroll
            for (int q = 0; q < SPW - 1; ++q)
#pragma unroll
                for (int i = q + 1; i < SPW; ++i) {
                    if constexpr (EXACT) {
#pragma clang fp contract(off)
                        u[i] = u[i] - urow[i][q] * u[q];
                    } else {
                        u[i] = fma(-urow[i][q], u[q], u[i]);
                    }
                }
#pragma unroll
            for (int i = 1; i < SPW; ++i) urow[i][SPW + lane] = u[i];
        }
        __syncthreads();
        if constexpr (EXACT) {
            // this thread's row, or with at most 64 rows row `lane` and every
            // NW-th group of columns
            constexpr int VL = 16 / (int)sizeof(T);
            typedef T vT __attribute__((ext_vector_type(VL)));
            const bool few = rows <= 64;
            const int row = few ? lane : tid;
            if (s_pos[row] >= cb + SPW) {
#pragma clang fp contract(off)
                T mult[SPW];
#pragma unroll
                for (int c = 0; c < SPW; ++c) mult[c] = tile[row][cb + c];
                for (int col = cb + SPW + (few ? wave * VL : 0); col < w; col += few ? NW * VL : VL) {
                    vT v = *reinterpret_cast<const vT *>(&tile[row][col]);
#pragma unroll
                    for (int c = 0; c < SPW; ++c) {
                        const vT u = *reinterpret_cast<const vT *>(&urow[c][col - cb]);
#pragma unroll
                        for (int e = 0; e < VL; ++e) v[e] = v[e] - mult[c] * u[e];
                    }
                    *reinterpret_cast<vT *>(&tile[row][col]) = v;
                }
            }
        } else {
            // this wave's 64 rows: A22 -= L21 U12, four independent 16 x 16 tiles
            // per 16 columns; rows already chosen keep their values
            const int lr = lane & 15, lk = lane >> 4;
            T af[4][4];
            int ps[4][4];
#pragma unroll
            for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    af[rt][s] = tile[wave * 64 + rt * 16 + lr][cb + 4 * s + lk];
                    ps[rt][s] = s_pos[wave * 64 + rt * 16 + Mfma<T>::row(lk, s)];
                }
            for (int ct = cb + SPW; ct < PNB; ct += 16) {
                T bf[4], cv[4][4];
#pragma unroll
                for (int s = 0; s < 4; ++s) bf[s] = urow[4 * s + lk][ct - cb + lr];
#pragma unroll
                for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) cv[rt][r] = tile[wave * 64 + rt * 16 + Mfma<T>::row(lk, r)][ct + lr];
                typename Mfma<T>::acc acc[4] = {};
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int rt = 0; rt < 4; ++rt) acc[rt] = Mfma<T>::op(af[rt][s], bf[s], acc[rt]);
#pragma unroll
                for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const T v = cv[rt][r] - acc[rt][r];
                        // (a chosen row is not even written: it may be taking its U12)
                        if (ps[rt][r] >= cb + SPW) tile[wave * 64 + rt * 16 + Mfma<T>::row(lk, r)][ct + lr] = v;
                    }
            }
        }
        // the pivot rows held here take their U12
        for (int i = wave; i < SPW; i += NW) {
            const int t = s_row[i];
            if (t >= 0 && cb + SPW + lane < PNB) tile[t][cb + SPW + lane] = urow[i][SPW + lane];
        }
        __syncthreads();
    }
    __syncthreads();

    if (g == 0) {
        if (tid < w) ipiv[k + tid] = (int64_t)k + s_piv[tid];
        if (tid == 0 && small < w && *info == (int64_t)n) *info = k + small;
    }
#pragma unroll 8
    for (int q = 0; q < PNB; ++q) {
        const int r = q * NW + wave;
        if (r < rows && lane < w) A[(long)(k + s_pos[r]) * lda + k + lane] = tile[r][lane];
    }
}

// ---------------------------------------------------------------- panels of up to 256 rows

// The panel A[k:k+m, k:k+w] with m <= 64 R <= 256, in FP64, by one workgroup:
// k_lu_panel's arithmetic (the same bits), but one wave holds 16 columns of all
// rows in registers, R rows per lane, so that a column needs no barrier and no LDS
// on its chain; a second wave solves the pivot rows' part right of the group
// meanwhile, and the four update the rest on the matrix cores.
//
// Bound by the chain of a column, 120 instructions of one wave for R = 1 and 400
// for R = 4.  A row per thread, with two LDS round trips and a barrier per column,
// took 68 us for any number of rows; this takes 34, 47, 57 and 68 us for R = 1 to
// 4 (an order of 256 is factored in 347 instead of 417 us).  One loop body for the
// 16 columns, the entries moving down a register per column, is 3 to 6 us slower:
// it eliminates more entries than there are.
constexpr size_t ONE_ROWS = 256;
template <int R> struct OneShared {
    double tile[R * 64 * PNB];           // see one_at
    double u[SPW][PNB - SPW];            // U12 of a group of columns
    unsigned long long act[R];           // rows not yet chosen
    int slot[PNB];                       // row of pivot j (-1: not known yet)
    int piv[PNB], pos[R * 64];
};
// Entry (row, col) of the tile: the 16-byte pieces of a row are permuted by its
// number, so that 16 consecutive rows read at one column touch all banks.
__device__ __forceinline__ int one_at(int row, int col) {
    return row * PNB + (((col >> 1) ^ (row & 15)) << 1) + (col & 1);
}
// Columns cb .. cb+15, by wave 0; pos[r] is the position of row 64 r + lane.  The
// pivot is the first maximum (see first_max_lane).  Every lane sets its best row's
// entries aside, and the winner's reach all lanes through scalar registers.  A
// chosen row's entries go to the tile when it is chosen (its registers are
// eliminated on, with a multiplier of zero), the others' multipliers column by
// column; then the row goes to sh.slot.
template <int R>
__device__ __forceinline__ void one_factor(OneShared<R> &sh, int cb, int w, int (&pos)[R]) {
    typedef double v2 __attribute__((ext_vector_type(2)));
    const int lane = opaque(threadIdx.x & 63);
    double x[R][SPW];
    unsigned long long act[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        act[r] = uniform(sh.act[r]);
#pragma unroll
        for (int q = 0; q < SPW; q += 2) {
            const v2 v = *reinterpret_cast<const v2 *>(&sh.tile[one_at(r * 64 + lane, cb + q)]);
            x[r][q] = v.x;
            x[r][q + 1] = v.y;
        }
    }
    static_for<SPW>([&](auto cc) __attribute__((always_inline)) {
        constexpr int c = decltype(cc)::value;
        const int j = cb + c;
        if (j >= w) return;
        unsigned key[R], d = 0u;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            key[r] = bit_of(act[r], rank_hi(fabs(x[r][c]), pos[r] == j), 0u);
            d = max(d, key[r]);
        }
        double y[SPW];  // the entries of this lane's best row, its number and position
        int best = 0, at = 0;
        auto aside = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int e = c; e < SPW; ++e) y[e] = x[0][e];
            best = 0;
            at = pos[0];
            unsigned most = key[0];
#pragma unroll
            for (int r = 1; r < R; ++r) {
                const bool up = key[r] > most;
#pragma unroll
                for (int e = c; e < SPW; ++e) y[e] = up ? x[r][e] : y[e];
                best = up ? r : best;
                at = up ? pos[r] : at;
                most = max(most, key[r]);
            }
        };
        d = dpp_max<DPP_SHR<1>>(d);
        d = dpp_max<DPP_SHR<2>>(d);
        d = dpp_max<DPP_SHR<4>>(d);
        d = dpp_max<DPP_SHR<8>>(d);
        d = dpp_max<DPP_BCAST15>(d);
        d = dpp_max<DPP_BCAST31>(d);
        const unsigned mx = lane_get(d, 63);
        aside();
        unsigned long long hit[R];
        int hits = 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            hit[r] = __ballot(key[r] == mx);
            hits += __popcll(hit[r]);
        }
        if (__builtin_expect(hits != 1, 0)) {  // equal high words: the low words, then the positions
            unsigned lo[R], ml = 0u;
            int mi = INT_MAX;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                lo[r] = key[r] == mx ? rank_lo(fabs(x[r][c])) : 0u;
                ml = max(ml, lo[r]);
            }
            ml = wave_max_u32(ml);
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (key[r] == mx && lo[r] == ml) mi = min(mi, pos[r]);
            mi = wave_min_i32(mi);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                key[r] = key[r] == mx && lo[r] == ml && pos[r] == mi ? 1u : 0u;
                hit[r] = __ballot(key[r] != 0u);
            }
            aside();
        }
        unsigned long long any = hit[0];
#pragma unroll
        for (int r = 1; r < R; ++r) any |= hit[r];
        const int l = __builtin_ctzll(any);
        double u[SPW];
#pragma unroll
        for (int e = c; e < SPW; ++e) u[e] = lane_get(y[e], l);
        const int t = lane_get(best, l) * 64 + l, pl = lane_get(at, l);
        if (lane == l) {
            if (c & 1) sh.tile[one_at(t, j)] = y[c];
#pragma unroll
            for (int e = (c + 1) & ~1; e < SPW; e += 2)
                *reinterpret_cast<v2 *>(&sh.tile[one_at(t, cb + e)]) = v2{y[e], y[e + 1]};
        }
        const double piv = u[c];
        const double rc = recip(piv);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            act[r] &= ~hit[r];
            pos[r] = pos[r] == pl ? j : (pos[r] == j ? pl : pos[r]);
            const double mult = div_recip(x[r][c], piv, rc);
            if (bit_of(act[r], true, false)) sh.tile[one_at(r * 64 + lane, j)] = mult;
            const double m = bit_of(act[r], mult, 0.0);
#pragma unroll
            for (int e = c + 1; e < SPW; ++e) x[r][e] = fma(-m, u[e], x[r][e]);
        }
        if (lane == 0) {
            sh.piv[j] = pl;
            __hip_atomic_store(&sh.slot[j], t, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    });
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) sh.act[r] = act[r];
    }
}

// U12 = L11^-1 A12 of columns cb .. cb+15, one column per lane, by another wave
// behind one_factor, which waits for nothing: the wait ends, and is bounded.
template <int R> __device__ __forceinline__ void one_solve(OneShared<R> &sh, int cb) {
    const int lane = opaque(threadIdx.x & 63);
    const int rest = PNB - SPW - cb, col = min(cb + SPW + lane, PNB - 1);
    double u12[SPW];
    static_for<SPW>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        int t = -1;
        for (int spin = 0; t == -1 && spin < (1 << 20); ++spin) {
            t = __hip_atomic_load(&sh.slot[cb + i], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (t == -1) __builtin_amdgcn_s_sleep(1);
        }
        const int r = max(__builtin_amdgcn_readfirstlane(t), 0);
        double l[SPW], v = sh.tile[one_at(r, col)];
#pragma unroll
        for (int q = 0; q < i; ++q) l[q] = sh.tile[one_at(r, cb + q)];
#pragma unroll
        for (int q = 0; q < i; ++q) v = fma(-l[q], u12[q], v);
        u12[i] = v;
        if (lane < rest) {
            sh.u[i][lane] = v;
            sh.tile[one_at(r, col)] = v;
        }
    });
}

template <int R>
__global__ __launch_bounds__(256) void k_lu_panel_one(double *__restrict__ A, long lda, int k, int m, int w,
                                                      int64_t *__restrict__ ipiv, int64_t *__restrict__ info, int n) {
    __shared__ __attribute__((aligned(16))) OneShared<R> sh;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    {   // all loads in flight before the LDS stores
        const int lane = tid & 63;
        constexpr int PER = R * 16;
        double v[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int r = q * 4 + wave;
            v[q] = (r < m && lane < w) ? A[(long)(k + r) * lda + k + lane] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < PER; ++q) sh.tile[one_at(q * 4 + wave, lane)] = v[q];  // zero past w and m
    }
    const unsigned long long have = __ballot(tid < m);
    if ((tid & 63) == 0 && wave < R) sh.act[wave] = have;
    if (tid < PNB) sh.slot[tid] = -1;
    __syncthreads();

    int pos[R];
#pragma unroll
    for (int r = 0; r < R; ++r) pos[r] = r * 64 + (tid & 63);
#pragma unroll 1
    for (int cb = 0; cb < w; cb += SPW) {
        if (wave == 0) one_factor(sh, cb, w, pos);
        else if (wave == 1 && cb + SPW < w) one_solve(sh, cb);
        __syncthreads();
        if (cb + SPW >= w) break;
        if (wave < R) {
            // this wave's 64 rows: A22 -= L21 U12; rows already chosen keep their values
            const int lane = opaque(tid & 63), lr = lane & 15, lk = lane >> 4;
            const unsigned long long act = uniform(sh.act[wave]);
            double af[4][4];
#pragma unroll
            for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                for (int s = 0; s < 4; ++s) af[rt][s] = sh.tile[one_at(wave * 64 + rt * 16 + lr, cb + 4 * s + lk)];
#pragma unroll 1
            for (int ct = cb + SPW; ct < PNB; ct += 16) {
                double bf[4], cv[4][4];
#pragma unroll
                for (int s = 0; s < 4; ++s) bf[s] = sh.u[4 * s + lk][ct - cb - SPW + lr];
#pragma unroll
                for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        cv[rt][r] = sh.tile[one_at(wave * 64 + rt * 16 + Mfma<double>::row(lk, r), ct + lr)];
                Mfma<double>::acc acc[4] = {};
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int rt = 0; rt < 4; ++rt) acc[rt] = Mfma<double>::op(af[rt][s], bf[s], acc[rt]);
#pragma unroll
                for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = rt * 16 + Mfma<double>::row(lk, r);
                        if ((act >> row) & 1ull) sh.tile[one_at(wave * 64 + row, ct + lr)] = cv[rt][r] - acc[rt][r];
                    }
            }
        }
        __syncthreads();
    }
    const int lane = opaque(tid & 63);
    if (wave == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) sh.pos[r * 64 + lane] = pos[r];
        // the first pivot below epsilon (every column has one: m >= w)
        const double d = lane < w ? sh.tile[one_at(sh.slot[lane], lane)] : 1.0;
        const unsigned long long small = __ballot(fabs(d) < eps_of<double>());
        if (lane == 0 && small != 0ull && *info == (int64_t)n) *info = k + __builtin_ctzll(small);
        if (lane < w) ipiv[k + lane] = (int64_t)k + sh.piv[lane];
    }
    __syncthreads();
#pragma unroll 8
    for (int q = 0; q < R * 16; ++q) {
        const int r = q * 4 + wave;
        if (r < m && lane < w) A[(long)(k + sh.pos[r]) * lda + k + lane] = sh.tile[one_at(r, lane)];
    }
}

// ---------------------------------------------------------------- row swaps

// Net effect of the swaps ipiv[k0 .. k0+cnt) as a list of (dst, src) rows:
// after the swaps, row dst holds what row src held before.  Swap s exchanges
// rows k0+s and p_s >= k0+s, so row k0+s is final after swap s and then
// holds what row p_s held just before it.  Before swap t, a row x >= k0+t
// holds what row k0+s held before swap s, for the last s < t with p_s = x,
// and its own content if there is none.  Following that rule back is one
// downward scan of the swaps from t-1, so every thread resolves its rows on
// its own: thread i the final content of row k0+i and, when swap i is the
// last to touch a row p_i beyond the block, that row's (what row k0+i held
// before swap i).  The list (block rows first) is written with ballot
// prefix counts.
// The scans read P eight entries at a time (one LDS latency per eight, not
// per entry); the entries are then tested in scan order.
__device__ __forceinline__ int swap_chase(const int *P, int k0, int x, int t) {
    int j = t - 1;
    for (; j >= 7; j -= 8) {
        int p[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q] = P[j - q];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (p[q] == x) x = k0 + (j - q);
    }
    for (; j >= 0; --j)
        if (P[j] == x) x = k0 + j;
    return x;
}
// True when no swap after t touches row x (P[t+1 .. cnt) != x).
__device__ __forceinline__ bool swap_last(const int *P, int x, int t, int cnt) {
    bool last = true;
    int j = t + 1;
    for (; j + 7 < cnt; j += 8) {
        int p[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q] = P[j + q];
#pragma unroll
        for (int q = 0; q < 8; ++q) last = last && p[q] != x;
    }
    for (; j < cnt; ++j) last = last && P[j] != x;
    return last;
}

// The list into LDS (dst[], src[]) by the 256 threads of a workgroup, in
// the order above; returns its length (at most 2 cnt).  P is scratch.
__device__ int swap_map_lds(const int64_t *__restrict__ ipiv, int k0, int cnt, int *P, int *dst,
                            int *src, int (*wcount)[SWB / 64]) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t < cnt) P[t] = (int)ipiv[k0 + t];
    __syncthreads();
    int src_in = k0 + t, dst_out = -1, src_out = -1;
    if (t < cnt) {
        const int pt = P[t];
        src_in = swap_chase(P, k0, pt, t);
        if (pt >= k0 + cnt && swap_last(P, pt, t, cnt)) {
            dst_out = pt;
            src_out = swap_chase(P, k0, k0 + t, t);
        }
    }
    const bool mv_in = t < cnt && src_in != k0 + t;
    const bool mv_out = dst_out >= 0 && src_out != dst_out;
    const unsigned long long b_in = __ballot(mv_in), b_out = __ballot(mv_out);
    if (lane == 0) { wcount[0][wave] = __popcll(b_in); wcount[1][wave] = __popcll(b_out); }
    __syncthreads();
    int off_in = 0, tot_in = 0, off_out = 0, tot_out = 0;
#pragma unroll
    for (int q = 0; q < SWB / 64; ++q) {
        if (q < wave) { off_in += wcount[0][q]; off_out += wcount[1][q]; }
        tot_in += wcount[0][q];
        tot_out += wcount[1][q];
    }
    if (mv_in) {
        const int at = off_in + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(b_in >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((unsigned)b_in, 0));
        dst[at] = k0 + t;
        src[at] = src_in;
    }
    if (mv_out) {
        const int at = tot_in + off_out +
                       (int)__builtin_amdgcn_mbcnt_hi((unsigned)(b_out >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((unsigned)b_out, 0));
        dst[at] = dst_out;
        src[at] = src_out;
    }
    __syncthreads();
    return tot_in + tot_out;
}

// Applies the swaps ipiv[k0 .. k0+cnt) (cnt <= SWB) to columns [c0, c1) and
// [c2, c3).  Every workgroup derives the row map itself (a few microseconds
// of its 256 threads, where a separate launch would cost more), then owns
// LCOLS columns: it reads every source row of the map, then writes the
// destinations, so the in-place permutation needs no ordering.
//
// Bound by memory: a row's 256 (FP32 128) bytes are read and written once.  All of
// a thread's entries are in flight together and stay in its registers: staged in
// LDS eight at a time, one workgroup filled a CU and 256 swaps of order 16384 took
// 67 us (FP32 39.5); this takes 34.5 (FP32 24.4).
constexpr int LCOLS = 32;
template <class T>
__global__ __launch_bounds__(SWB) void k_laswp(T *__restrict__ A, long lda, const int64_t *__restrict__ ipiv,
                                               int k0, int cnt_sw, int c0, int c1, int c2, int c3) {
    constexpr int RG = SWB / LCOLS, PER = 2 * SWB / RG, B = 8;  // row groups, entries per thread, per test
    __shared__ int dst[2 * SWB], src[2 * SWB];
    __shared__ long to[2 * SWB], from[2 * SWB];  // their offsets
    __shared__ int P[SWB];
    __shared__ int wcount[2][SWB / 64];
    const int cnt = __builtin_amdgcn_readfirstlane(swap_map_lds(ipiv, k0, cnt_sw, P, dst, src, wcount));
    if (cnt == 0) return;
    for (int i = threadIdx.x; i < cnt; i += SWB) {
        to[i] = (long)dst[i] * lda;
        from[i] = (long)src[i] * lda;
    }
    __syncthreads();
    // column block -> absolute columns (past the last: the first, not written)
    const int w1 = c1 - c0, lc = blockIdx.x * LCOLS + (int)threadIdx.x % LCOLS, rg = threadIdx.x / LCOLS;
    const bool okc = lc < w1 + (c3 - c2);
    T *const a = A + (lc < w1 ? c0 + lc : okc ? c2 + (lc - w1) : w1 > 0 ? c0 : c2);
    T v[PER];
#pragma unroll
    for (int b = 0; b < PER; b += B)
        if (b * RG < cnt) {
#pragma unroll
            for (int q = b; q < b + B; ++q) v[q] = a[from[min(rg + q * RG, cnt - 1)]];
        }
    // every value has arrived before the barrier
#pragma unroll
    for (int b = 0; b < PER; b += B)
        if (b * RG < cnt) {
#pragma unroll
            for (int q = b; q < b + B; ++q) asm volatile("" : "+v"(v[q]));
        }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < PER; b += B)
        if (b * RG < cnt) {
#pragma unroll
            for (int q = b; q < b + B; ++q)
                if (okc && rg + q * RG < cnt) a[to[rg + q * RG]] = v[q];
        }
}

// ---------------------------------------------------------------- TRSM

// The block-row solve B := L^-1 B of a factored panel, with L the unit-lower
// jb x jb block A[j0:j0+jb, j0:j0+jb] (jb <= 64) and B = A[j0:j0+jb, c0:c1)
// (the reference applies the same elimination to these columns row by row,
// lu.rs:603-616), is done as a product with L^-1: the inverse is formed once
// per panel, and every 64-column slab of B is then one 64-deep matrix-core
// product instead of a 64-step dependent sweep.  L has a unit diagonal and,
// under partial pivoting, entries of magnitude at most 1.

// B := inv * B for one 64-column slab per workgroup, in place: the slab is
// read whole into LDS before any of it is written.  Wave w computes rows
// [16 w, 16 w + 16) of the slab as four 16 x 16 accumulators over 16 k-steps.
template <class T>
__global__ __launch_bounds__(256) void k_trsm_llu(T *__restrict__ A, long lda, int j0, int jb, int c0,
                                                  int c1, const T *__restrict__ inv) {
    using Acc = typename Mfma<T>::acc;
    __shared__ T Li[PNB][PNB + 1];  // Li[k][i] = inv[i][k]
    __shared__ T X[PNB][PNB + 1];   // X[k][c] = B[k][c]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int cb = c0 + blockIdx.x * 64;
    const int nc = min(64, c1 - cb);
    {
        constexpr int PER = PNB * PNB / 256;
        T vl[PER], vx[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = q * 256 + tid, r = e >> 6, c = e & 63;
            vl[q] = inv[e];
            vx[q] = (r < jb && c < nc) ? A[(long)(j0 + r) * lda + cb + c] : T(0);
        }
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = q * 256 + tid, r = e >> 6, c = e & 63;
            Li[c][r] = vl[q];
            X[r][c] = vx[q];
        }
    }
    __syncthreads();
    Acc acc[4];
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) acc[jc] = Acc{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < PNB / 4; ++s) {
        const T a = Li[4 * s + lk][16 * wave + lr];
#pragma unroll
        for (int jc = 0; jc < 4; ++jc) acc[jc] = Mfma<T>::op(a, X[4 * s + lk][16 * jc + lr], acc[jc]);
    }
#pragma unroll
    for (int jc = 0; jc < 4; ++jc)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * wave + Mfma<T>::row(lk, r), col = 16 * jc + lr;
            if (row < jb && col < nc) A[(long)(j0 + row) * lda + cb + col] = acc[jc][r];
        }
}

// ---------------------------------------------------------------- driver

// The step between an inner panel and its update, for the other columns of the
// outer block: the panel's swaps on columns [c0, c1) and [c2, c3), the inverse of
// its unit-lower block, and the block-row solve B := L^-1 B on the swapped rows
// of [c2, c3).  A workgroup owns 32 columns on one side (at least one workgroup
// has the right side, if that inverse is needed): it reads every row its columns
// move, then writes them.  Wave 0 derives the row moves while wave 1 inverts the
// diagonal blocks; every workgroup on the right forms the whole inverse, and the
// first stores it for the outer block row (have_inv: it is there already).
//
// Bound by latencies: four dependent trips to memory and about 4,000 cycles of
// inversion and product.  It takes 17 us in FP64 (12 in FP32) on average at order
// 16384, where three launches, for the inverse, the swaps and the solve,
// took 8.5, 13.6 and 8.
//
// L^-1 in blocks: the diagonal ones of IB x IB by forward substitution, a lane
// per column, then X21 = -X22 (L21 X11) by doubling sizes on the matrix cores.
// IB is 16 in FP64 (a shorter chain) and 32 in FP32, which keeps the values that
// the low-precision factorizations were tested with.
template <class T> struct InvBlock { static constexpr int value = 16; };
template <> struct InvBlock<float> { static constexpr int value = 32; };
constexpr int RCOLS = 32;  // columns per workgroup
template <class T>
__global__ __launch_bounds__(256) void k_row_step(T *__restrict__ A, long lda, const int64_t *__restrict__ ipiv,
                                                  int j0, int jb, int c0, int c1, int c2, int c3, T *inv,
                                                  int have_inv) {
    using Acc = typename Mfma<T>::acc;
    constexpr int IB = InvBlock<T>::value, LD = PNB + TilePad<T>::value;
    __shared__ __attribute__((aligned(16))) T L[PNB][LD];  // L, overwritten by L^-1 block by block
    __shared__ T Tm[PNB / 2][PNB / 2 + 1];                 // L21 X11
    __shared__ T X[PNB][RCOLS + 1];
    __shared__ int P[PNB], src_in[PNB], dst_out[PNB], src_out[PNB], s_out;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int left = (c1 - c0 + RCOLS - 1) / RCOLS;
    const bool right = (int)blockIdx.x >= left;
    const int cb = right ? c2 + ((int)blockIdx.x - left) * RCOLS : c0 + (int)blockIdx.x * RCOLS;
    const int ce = min(cb + RCOLS, right ? c3 : c1);

    if (tid < jb) P[tid] = (int)ipiv[j0 + tid];
    if (right) {
        constexpr int PER = PNB * PNB / 256;
        T v[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int r = q * 4 + wave, c = lane;
            v[q] = have_inv ? inv[r * PNB + c] : (r < jb && c < r) ? A[(long)(j0 + r) * lda + j0 + c] : T(0);
        }
#pragma unroll
        for (int q = 0; q < PER; ++q) L[q * 4 + wave][lane] = v[q];
    }
    __syncthreads();
    if (wave == 0) {
        // the final content of row j0 + lane, and of the row that swap `lane`
        // is the last to touch beyond the block
        int so = -1, pt = -1;
        bool mv = false;
        if (lane < jb) {
            pt = P[lane];
            src_in[lane] = swap_chase(P, j0, pt, lane);
            if (pt >= j0 + jb && swap_last(P, pt, lane, jb)) {
                so = swap_chase(P, j0, j0 + lane, lane);
                mv = so != pt;
            }
        }
        const unsigned long long b = __ballot(mv);
        if (mv) {
            const int at = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b, 0));
            dst_out[at] = pt;
            src_out[at] = so;
        }
        if (lane == 0) s_out = __popcll(b);
    } else if (wave == 1 && right && !have_inv) {
        // every read of a block precedes the wave's writes to it
        const int o = lane / IB * IB, j = lane % IB;
        T x[IB];
#pragma unroll
        for (int i = 0; i < IB; ++i) {
            T s = (i == j) ? T(1) : T(0);
#pragma unroll
            for (int q = 0; q < i; ++q) s -= L[o + i][o + q] * x[q];
            x[i] = s;
        }
#pragma unroll
        for (int i = 0; i < IB; ++i) L[o + i][o + j] = x[i];  // zero above the diagonal
    }
    __syncthreads();

    // the rows: element (q * 8 + tid / 32, tid % 32) of the block's and of the others
    constexpr int RG = 256 / RCOLS, PER = PNB / RG;
    const int rg = tid / RCOLS, cl = tid % RCOLS, col = cb + cl;
    const int outs = s_out;
    T vi[PER], vo[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int i = q * RG + rg;
        vi[q] = i < jb && col < ce ? A[(long)src_in[i] * lda + col] : T(0);
        vo[q] = i < outs && col < ce ? A[(long)src_out[i] * lda + col] : T(0);
    }
    if (right && !have_inv) {
        if constexpr (IB == 16) {
            const int o = wave * 32;
            const bool on = wave < 2;
            if (on) {
                Acc acc = Acc{0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = Mfma<T>::op(L[o + 16 + lr][o + 4 * s + lk], L[o + 4 * s + lk][o + lr], acc);
#pragma unroll
                for (int r = 0; r < 4; ++r) Tm[16 * wave + Mfma<T>::row(lk, r)][lr] = acc[r];
            }
            __syncthreads();
            if (on) {
                Acc acc = Acc{0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = Mfma<T>::op(L[o + 16 + lr][o + 16 + 4 * s + lk], Tm[16 * wave + 4 * s + lk][lr], acc);
#pragma unroll
                for (int r = 0; r < 4; ++r) L[o + 16 + Mfma<T>::row(lk, r)][o + lr] = -acc[r];
            }
            __syncthreads();
        }
        constexpr int H = PNB / 2;
        const int tr = (wave >> 1) * 16, tc = (wave & 1) * 16;  // this wave's 16 x 16 tile
        {   // Tm = L21 X11
            Acc acc = Acc{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < H / 4; ++s) acc = Mfma<T>::op(L[H + tr + lr][4 * s + lk], L[4 * s + lk][tc + lr], acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) Tm[tr + Mfma<T>::row(lk, r)][tc + lr] = acc[r];
        }
        __syncthreads();
        {   // X21 = -X22 Tm, over L21 (no longer read)
            Acc acc = Acc{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < H / 4; ++s)
                acc = Mfma<T>::op(L[H + tr + lr][H + 4 * s + lk], Tm[4 * s + lk][tc + lr], acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) L[H + tr + Mfma<T>::row(lk, r)][tc + lr] = -acc[r];
        }
        __syncthreads();
        // the rows and columns past jb were staged as zeros: they inverted to the
        // identity, and become zeros again
#pragma unroll
        for (int q = 0; q < PNB * PNB / 256; ++q) {
            const int i = q * 4 + wave, c = lane;
            const T v = i < jb && c < jb && c <= i ? L[i][c] : T(0);
            L[i][c] = v;
            if ((int)blockIdx.x == left) inv[i * PNB + c] = v;
        }
    }
    if (right) {
#pragma unroll
        for (int q = 0; q < PER; ++q) X[q * RG + rg][cl] = vi[q];
    }
    __syncthreads();  // every row has been read
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int i = q * RG + rg;
        if (!right && i < jb && col < ce && src_in[i] != j0 + i) A[(long)(j0 + i) * lda + col] = vi[q];
        if (i < outs && col < ce) A[(long)dst_out[i] * lda + col] = vo[q];
    }
    if (!right) return;
    // wave w: rows [16 w, 16 w + 16) of L^-1 B as two 16 x 16 tiles
    Acc acc[2] = {};
#pragma unroll
    for (int s = 0; s < PNB / 4; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t)
            acc[t] = Mfma<T>::op(L[16 * wave + lr][4 * s + lk], X[4 * s + lk][16 * t + lr], acc[t]);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * wave + Mfma<T>::row(lk, r), c = cb + 16 * t + lr;
            if (row < jb && c < ce) A[(long)(j0 + row) * lda + c] = acc[t][r];
        }
}

// Set by lu_factor_lowp for its duration: FP32 panels are then factored with
// tournament pivoting (tslu.hip) in this workspace.
static thread_local void *g_tslu_work = nullptr;

template <class T>
static int panel(hipStream_t s, T *a, size_t lda, size_t k, size_t m, size_t w, int64_t *ipiv,
                 int64_t *info, size_t n, const LuWork &lw);

template <class T>
static T *linv_of(const LuWork &lw, size_t j0);

// The panel by tournament pivoting when lu_factor_lowp asked for it (the
// tournament also writes L11^-1: *linv_done), else by partial pivoting.
template <class T>
static int panel_any(hipStream_t s, T *a, size_t lda, size_t k, size_t m, size_t w, int64_t *ipiv,
                     int64_t *info, size_t n, const LuWork &lw, bool *linv_done) {
    *linv_done = false;
    if constexpr (std::is_same<T, float>::value) {
        if (g_tslu_work && m <= tslu_max_rows(n)) {
            *linv_done = true;
            return tslu_panel(s, a, lda, k, m, w, ipiv, info, n, g_tslu_work, linv_of<float>(lw, k));
        }
    }
    return panel<T>(s, a, lda, k, m, w, ipiv, info, n, lw);
}

// Largest panel height: the panel's workgroups exchange data while they run,
// so all of them must be resident at once, and their slots must fit the
// exchange area.  The bound is the device's occupancy for this kernel (one
// workgroup per CU: its LDS tile takes most of the CU's LDS) times its CUs.
template <class T>
static int panel_rows_max(size_t *out) {
    Device *d = nullptr;
    RLG_TRY(current_device(&d));
    static thread_local int per_cu[2] = {-1, -1};
    int &bpc = per_cu[sizeof(T) == 8];
    if (bpc < 0)
        RLG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &bpc, reinterpret_cast<const void *>(k_lu_panel<T, sizeof(T) == 4>), PanelRows<T>::value, 0));
    size_t g = (size_t)bpc * (size_t)d->num_cus;
    if (g > (size_t)GMAX) g = GMAX;
    *out = g * PanelRows<T>::value;
    return RLG_OK;
}

template <class T>
static int panel(hipStream_t s, T *a, size_t lda, size_t k, size_t m, size_t w, int64_t *ipiv,
                 int64_t *info, size_t n, const LuWork &lw) {
    size_t mmax = 0;
    RLG_TRY(panel_rows_max<T>(&mmax));
    if (m > mmax) {
        set_error("LU panel of %zu rows exceeds the %zu rows that this device's CUs hold", m, mmax);
        return RLG_E_INVALID_ARG;
    }
    const unsigned G = ceil_div(m, PanelRows<T>::value);
    // algorithmic bytes: the m x w panel read once and written once
    RLG_PROF_W("lu_panel", s, 2.0 * (double)m * (double)w * sizeof(T));
    constexpr unsigned PT = PanelRows<T>::value;
    constexpr bool EX = sizeof(T) == 4;
    if constexpr (!EX) {
        // one workgroup: the fewer rows per lane, the shorter the chain (see the kernel)
        if (m <= ONE_ROWS && n > (size_t)PNB) {
            auto one = [&](auto rows) {
                hipLaunchKernelGGL((k_lu_panel_one<decltype(rows)::value>), dim3(1), dim3(256), 0, s, a, (long)lda,
                                   (int)k, (int)m, (int)w, ipiv, info, (int)n);
            };
            if (m <= 64) one(std::integral_constant<int, 1>{});
            else if (m <= 128) one(std::integral_constant<int, 2>{});
            else if (m <= 192) one(std::integral_constant<int, 3>{});
            else one(std::integral_constant<int, 4>{});
            RLG_LAUNCHED();
            return RLG_OK;
        }
    }
    if (G == 1) {  // no exchange; in FP64 the whole matrix (n <= 64), to the reference's bits
        hipLaunchKernelGGL((k_lu_panel<T, true>), dim3(1), dim3(PT), 0, s, a, (long)lda, (int)k, (int)m, (int)w,
                           ipiv, info, (int)n, lw.xch, lw.timeout);
        RLG_LAUNCHED();
        return RLG_OK;
    }
    // A cooperative launch: the runtime starts the grid only with every
    // workgroup resident at once (and refuses a grid that cannot be), which
    // the per-column exchange between workgroups relies on.
    T *a_ = a;
    long lda_ = (long)lda;
    int k_ = (int)k, m_ = (int)m, w_ = (int)w, n_ = (int)n;
    xword *xch_ = lw.xch;
    int *to_ = lw.timeout;
    void *args[] = {&a_, &lda_, &k_, &m_, &w_, &ipiv, &info, &n_, &xch_, &to_};
    RLG_HIP(hipLaunchCooperativeKernel(reinterpret_cast<const void *>(k_lu_panel<T, EX>), dim3(G), dim3(PT),
                                       args, 0, s));
    return RLG_OK;
}

template <class T>
static int laswp(hipStream_t s, T *a, size_t lda, const int64_t *ipiv, size_t k0, size_t cnt,
                 size_t c0, size_t c1, size_t c2, size_t c3) {
    const size_t ncols = (c1 - c0) + (c3 - c2);
    if (ncols == 0 || cnt == 0) return RLG_OK;
    // a longer sequence is applied SWB swaps at a time, in order: the same
    // sequence of transpositions
    for (size_t off = 0; off < cnt; off += SWB) {
        const size_t c = cnt - off < (size_t)SWB ? cnt - off : SWB;
        // algorithmic bytes: at most 2 c rows change, each read and written
        RLG_PROF_W("laswp", s, 2.0 * 2.0 * (double)c * (double)ncols * sizeof(T));
        hipLaunchKernelGGL(k_laswp<T>, dim3(ceil_div(ncols, LCOLS)), dim3(SWB), 0, s, a, (long)lda,
                           ipiv, (int)(k0 + off), (int)c, (int)c0, (int)c1, (int)c2, (int)c3);
        RLG_LAUNCHED();
    }
    return RLG_OK;
}

// The inverse of panel j0's unit-lower block: slot (j0 mod ONB) / PNB of the
// outer block's inverses.
template <class T>
static T *linv_of(const LuWork &lw, size_t j0) {
    return static_cast<T *>(lw.linv) + ((j0 % ONB) / PNB) * PNB * PNB;
}

template <class T>
static int row_step(hipStream_t s, T *a, size_t lda, const int64_t *ipiv, size_t n, size_t j0, size_t jb, size_t c0,
                    size_t c3, const LuWork &lw, bool have_inv) {
    const size_t left = ceil_div(j0 - c0, RCOLS), right = ceil_div(c3 - j0 - jb, RCOLS);
    // the last panel's inverse has no use; others' serve the outer block row too
    const size_t blocks = left + (right || j0 + jb == n || have_inv ? right : 1);
    if (blocks == 0) return RLG_OK;
    // algorithmic bytes: at most 2 jb rows of these columns read and written, the
    // block read and its inverse written
    RLG_PROF_W("row_step", s, (4.0 * (double)jb * (double)(c3 - c0 - jb) + 2.0 * PNB * PNB) * sizeof(T));
    hipLaunchKernelGGL(k_row_step<T>, dim3((unsigned)blocks), dim3(256), 0, s, a, (long)lda, ipiv, (int)j0, (int)jb,
                       (int)c0, (int)j0, (int)(j0 + jb), (int)c3, linv_of<T>(lw, j0), (int)have_inv);
    RLG_LAUNCHED();
    return RLG_OK;
}

template <class T>
static int trsm_llu(hipStream_t s, T *a, size_t lda, size_t j0, size_t jb, size_t c0, size_t c1,
                    const LuWork &lw) {
    if (c1 <= c0 || jb <= 1) return RLG_OK;
    // algorithmic bytes: the 64 x 64 inverse and the jb x (c1-c0) block row (read + write)
    RLG_PROF_W("trsm", s, ((double)PNB * PNB + 2.0 * (double)jb * (double)(c1 - c0)) * sizeof(T));
    hipLaunchKernelGGL(k_trsm_llu<T>, dim3(ceil_div(c1 - c0, 64)), dim3(256), 0, s, a, (long)lda,
                       (int)j0, (int)jb, (int)c0, (int)c1, (const T *)linv_of<T>(lw, j0));
    RLG_LAUNCHED();
    return RLG_OK;
}

template <class T>
using UpdateFn = int (*)(hipStream_t, size_t, size_t, size_t, const T *, size_t, const T *, size_t,
                         T *, size_t);

// C -= A * B in working precision.
template <class T>
static int update_native(hipStream_t s, size_t m, size_t n, size_t k, const T *a, size_t lda,
                         const T *b, size_t ldb, T *c, size_t ldc) {
    return gemm_t<T>(s, m, n, k, T(-1), a, lda, b, ldb, T(1), c, ldc);
}

// set by lu_factor_lowp for its duration: precision and the packed-operand
// areas (one for the caller's stream, one for the look-ahead's second stream)
static thread_local int g_lowp_prec = RLG_PREC_F16;
static thread_local void *g_lowp_pack = nullptr;
static thread_local void *g_lowp_pack2 = nullptr;
static thread_local size_t g_lowp_pack_bytes = 0;
static int update_lowp(hipStream_t s, size_t m, size_t n, size_t k, const float *a, size_t lda,
                       const float *b, size_t ldb, float *c, size_t ldc) {
    return gemm_lowp(s, g_lowp_prec, m, n, k, -1.f, a, lda, b, ldb, 1.f, c, ldc, false, false,
                     g_lowp_pack, g_lowp_pack_bytes);
}

// The look-ahead's update on the second stream.  Its workgroups reserve LDS
// they do not use, so that one of them and one workgroup of the panel chain
// (tournament, row swaps, block-row solve, depth-64 update: at most 70 KB)
// share a CU, where two of them would fill its 160 KB: the split FP16
// kernel stages 80 KB, the FP32 one 66 KB.
constexpr size_t LU_SPLIT_PAD = 8 << 10, LU_F32_PAD = 24 << 10;
constexpr size_t LOOKAHEAD_MIN_N = 8192;  // smallest order factored with look-ahead
static int update_lowp_aux(hipStream_t s, size_t m, size_t n, size_t k, const float *a, size_t lda,
                           const float *b, size_t ldb, float *c, size_t ldc) {
    return gemm_lowp(s, g_lowp_prec, m, n, k, -1.f, a, lda, b, ldb, 1.f, c, ldc, false, false,
                     g_lowp_pack2, g_lowp_pack_bytes, LU_SPLIT_PAD);
}
static int update_f32_aux(hipStream_t s, size_t m, size_t n, size_t k, const float *a, size_t lda,
                          const float *b, size_t ldb, float *c, size_t ldc) {
    return gemm_t_padded<float>(s, m, n, k, -1.f, a, lda, b, ldb, 1.f, c, ldc, false, false, LU_F32_PAD);
}

// Events used to order the look-ahead stream against the main stream.
struct StepEvents {
    hipEvent_t ready = nullptr, big = nullptr;
    bool big_pending = false;
    ~StepEvents() {
        if (ready) (void)hipEventDestroy(ready);
        if (big) (void)hipEventDestroy(big);
    }
};

// Factor the outer block of columns [k0, k0+kb): inner panels of PNB columns,
// their swaps on the rest of the block, and the block-local updates.
template <class T>
static int outer_panel(hipStream_t s, size_t n, T *a, size_t lda, int64_t *ipiv, int64_t *info,
                       const LuWork &lw, size_t k0, size_t kb) {
    for (size_t j0 = k0; j0 < k0 + kb; j0 += PNB) {
        const size_t jb = k0 + kb - j0 < (size_t)PNB ? k0 + kb - j0 : PNB;
        bool linv_done = false;
        RLG_TRY(panel_any<T>(s, a, lda, j0, n - j0, jb, ipiv, info, n, lw, &linv_done));
        // swaps and block-row solve on the other columns of the outer block
        RLG_TRY(row_step<T>(s, a, lda, ipiv, n, j0, jb, k0, k0 + kb, lw, linv_done));
        if (j0 + jb < k0 + kb) {
            RLG_TRY(update_native<T>(s, n - j0 - jb, k0 + kb - j0 - jb, jb, a + (j0 + jb) * lda + j0,
                                     lda, a + j0 * lda + j0 + jb, lda, a + (j0 + jb) * lda + j0 + jb,
                                     lda));
        }
    }
    return RLG_OK;
}

// Right-looking blocked LU, with look-ahead when `aux_update` is given.
// After outer block k is factored and its block row solved, the trailing
// update is split: the columns of block k+1 are updated first on the
// caller's stream, which then factors block k+1, while the rest of the
// trailing update runs on a second stream (`aux_update`; a stream created
// for the call, default priority).  The next step's row swaps and
// block-row solve wait for that update on an event.  The two streams touch
// disjoint columns meanwhile (block k+1's own panels, swaps and updates stay
// inside its columns), every entry receives the same updates in the same
// order, and the split follows the update's 128-wide tile grid, so the
// factors are the same as without look-ahead.
//
// Look-ahead is used with the tournament panels only.  Their workgroups
// never wait for one another, so they run beside the update on whatever
// CUs are free.  The partial-pivoting panel is a cooperative launch, which
// the runtime does not overlap with other streams' kernels.  An earlier form
// with a non-cooperative exchange panel beside the second stream stalled on
// the GPU.
template <class T>
static int lu_factor_impl(hipStream_t s, size_t n, T *a, size_t lda, int64_t *ipiv, int64_t *info,
                          void *work, UpdateFn<T> big_update, UpdateFn<T> aux_update) {
    // Below this order factorizations are mostly run several at a time (the
    // serving loop's systems go up to order 4096), and those already share
    // the device: there a second stream per factorization measured slower
    // (1,450 -> 975 solves/s at 2,000 requests/s offered).
    LuWork lw = carve(work, n, sizeof(T));
    // exchange tags restart with every factorization
    RLG_TRY(fill_u32(reinterpret_cast<uint32_t *>(lw.xch), 2 * xch_words(sizeof(T)), 0u, s));
    RLG_TRY(fill_u32(reinterpret_cast<uint32_t *>(lw.timeout), 1, 0u, s));
    RLG_TRY(fill_i64(info, 1, (int64_t)n, s));
    if (n == 0) return RLG_OK;
    AuxStream aux;
    hipStream_t s2 = nullptr;
    StepEvents ev;
    if (aux_update && n >= LOOKAHEAD_MIN_N) {
        RLG_TRY(aux.create());
        s2 = aux.s;
        RLG_HIP(hipEventCreateWithFlags(&ev.ready, hipEventDisableTiming));
        RLG_HIP(hipEventCreateWithFlags(&ev.big, hipEventDisableTiming));
    }
    RLG_TRY(outer_panel<T>(s, n, a, lda, ipiv, info, lw, 0, n < (size_t)ONB ? n : ONB));
    for (size_t k0 = 0; k0 < n; k0 += ONB) {
        const size_t kb = n - k0 < (size_t)ONB ? n - k0 : ONB;
        const size_t c0 = k0 + kb;
        if (ev.big_pending) {  // the previous trailing update must be complete
            RLG_HIP(hipStreamWaitEvent(s, ev.big, 0));
            ev.big_pending = false;
        }
        // outer swaps on everything left and right of the outer block
        RLG_TRY(laswp<T>(s, a, lda, ipiv, k0, kb, 0, k0, c0, n));
        if (c0 >= n) break;
        for (size_t j0 = k0; j0 < c0; j0 += PNB) {
            const size_t jb = c0 - j0 < (size_t)PNB ? c0 - j0 : PNB;
            RLG_TRY(trsm_llu<T>(s, a, lda, j0, jb, c0, n, lw));
            if (j0 + jb < c0)
                RLG_TRY(update_native<T>(s, c0 - j0 - jb, n - c0, jb, a + (j0 + jb) * lda + j0, lda,
                                         a + j0 * lda + c0, lda, a + (j0 + jb) * lda + c0, lda));
        }
        const size_t kb2 = n - c0 < (size_t)ONB ? n - c0 : ONB;
        if (!s2 || c0 + kb2 >= n) {
            RLG_TRY(big_update(s, n - c0, n - c0, kb, a + c0 * lda + k0, lda, a + k0 * lda + c0, lda,
                               a + c0 * lda + c0, lda));
        } else {
            // look-ahead columns first, then the rest on the second stream
            RLG_TRY(big_update(s, n - c0, kb2, kb, a + c0 * lda + k0, lda, a + k0 * lda + c0, lda,
                               a + c0 * lda + c0, lda));
            RLG_HIP(hipEventRecord(ev.ready, s));
            RLG_HIP(hipStreamWaitEvent(s2, ev.ready, 0));
            RLG_TRY(aux_update(s2, n - c0, n - c0 - kb2, kb, a + c0 * lda + k0, lda,
                               a + k0 * lda + c0 + kb2, lda, a + c0 * lda + c0 + kb2, lda));
            RLG_HIP(hipEventRecord(ev.big, s2));
            ev.big_pending = true;
        }
        RLG_TRY(outer_panel<T>(s, n, a, lda, ipiv, info, lw, c0, kb2));
    }
    if (ev.big_pending) RLG_HIP(hipStreamWaitEvent(s, ev.big, 0));
    return RLG_OK;
}

template <class T>
int lu_factor(hipStream_t s, size_t n, T *a, size_t lda, int64_t *ipiv, int64_t *info, void *work) {
    return lu_factor_impl<T>(s, n, a, lda, ipiv, info, work, &update_native<T>, nullptr);
}
template int lu_factor<double>(hipStream_t, size_t, double *, size_t, int64_t *, int64_t *, void *);
template int lu_factor<float>(hipStream_t, size_t, float *, size_t, int64_t *, int64_t *, void *);

// The trailing updates are at most n x n with depth ONB; the look-ahead's
// second stream has a packed-operand area of its own.
size_t lu_lowp_work_bytes(size_t n) {
    return align_up(lu_work_bytes(n, 4)) + 2 * align_up(gemm_lowp_pack_bytes(n, n, ONB)) +
           tslu_work_bytes(n);
}

int lu_factor_lowp(hipStream_t s, int prec, int pivot, size_t n, float *a, size_t lda, int64_t *ipiv,
                   int64_t *info, void *work) {
    char *w = static_cast<char *>(work);
    const size_t pack = align_up(gemm_lowp_pack_bytes(n, n, ONB));
    g_lowp_prec = prec;
    g_lowp_pack = w + align_up(lu_work_bytes(n, 4));
    g_lowp_pack2 = static_cast<char *>(g_lowp_pack) + pack;
    g_lowp_pack_bytes = gemm_lowp_pack_bytes(n, n, ONB);
    g_tslu_work = nullptr;
    int st = RLG_OK;
    UpdateFn<float> aux = nullptr;
    if (pivot == RLG_PIVOT_TOURNAMENT) {
        g_tslu_work = static_cast<char *>(g_lowp_pack2) + pack;
        st = tslu_reset(s, g_tslu_work, n);
        aux = prec == RLG_PREC_F32 ? &update_f32_aux : &update_lowp_aux;
    }
    if (st == RLG_OK)
        st = lu_factor_impl<float>(s, n, a, lda, ipiv, info, work,
                                   prec == RLG_PREC_F32 ? &update_native<float> : &update_lowp, aux);
    g_lowp_pack = nullptr;
    g_lowp_pack2 = nullptr;
    g_lowp_pack_bytes = 0;
    g_tslu_work = nullptr;
    return st;
}

// ---------------------------------------------------------------- solve

// tmp[r][k] = b[r][raw[k]]: y = P b with (P b)[k] = b[raw[k]], which is the
// reference's permute_vector_into_buffer (permutation_matrix.rs:369-382)
// applied with the stored inverse permutation.
template <class T>
__global__ void k_gather_rows(size_t n, size_t nrhs, const int64_t *__restrict__ raw,
                              const T *__restrict__ b, size_t ldb, T *__restrict__ y, size_t ldy) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t r = blockIdx.y;
    if (i < n && r < nrhs) y[r * ldy + i] = b[r * ldb + raw[i]];
}

template <class T>
int lu_solve(hipStream_t s, size_t n, const T *lu, size_t lda, const int64_t *raw, size_t nrhs,
             const T *b, size_t ldb, T *x, size_t ldx, T *tmp) {
    if (n == 0 || nrhs == 0) return RLG_OK;
    // y = P b, then L^-1 y, then U^-1 of that, each into the buffer the one
    // before does not use; with x and b apart the last lands in x by itself
    const bool apart = !vectors_overlap(n, nrhs, b, ldb, x, ldx);
    T *y = apart ? x : tmp, *z = apart ? tmp : x;
    const size_t ldy = apart ? ldx : n, ldz = apart ? n : ldx;
    {
        RLG_PROF("gather", s);
        hipLaunchKernelGGL(k_gather_rows<T>, dim3(ceil_div(n, 256), (unsigned)nrhs), dim3(256), 0, s, n,
                           nrhs, raw, b, ldb, y, ldy);
        RLG_LAUNCHED();
    }
    RLG_TRY(trsv_lower<T>(s, n, lu, lda, true, nrhs, y, ldy, z, ldz));
    RLG_TRY(trsv_upper<T>(s, n, lu, lda, nrhs, z, ldz, y, ldy));
    if (!apart)
        RLG_HIP(hipMemcpy2DAsync(x, ldx * sizeof(T), tmp, n * sizeof(T), n * sizeof(T), nrhs,
                                 hipMemcpyDeviceToDevice, s));
    return RLG_OK;
}
template int lu_solve<double>(hipStream_t, size_t, const double *, size_t, const int64_t *, size_t,
                              const double *, size_t, double *, size_t, double *);
template int lu_solve<float>(hipStream_t, size_t, const float *, size_t, const int64_t *, size_t,
                             const float *, size_t, float *, size_t, float *);

}  // namespace rlg
