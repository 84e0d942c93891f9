// Tournament pivoting (TSLU, the panel step of CALU: Grigori, Demmel and
// Xiang, SIAM J. Matrix Anal. Appl. 32 (2011)) for the FP32 panels of the
// mixed-precision LU.  The plain FP64 drop-in keeps the reference's partial
// pivoting (lu.hip); the mixed factorization only has to be stable enough for
// iterative refinement, which TSLU is in practice (its growth factor behaves
// like partial pivoting's), and it needs a few reduction levels per panel
// instead of one grid-wide exchange per column.
//
// Two launches factor the m x w panel A[k:k+m, k:k+w] (w <= 64):
//
// k_tslu_tourney, one 256-thread workgroup per 256-row leaf:
//   1. each workgroup runs partial pivoting on its leaf and writes the row
//      numbers of its w winners;
//   2. every tree node merges up to four children: the workgroup that
//      completes the last child (an atomic arrival count per node) loads the
//      children's winners' original rows and runs partial pivoting on those
//      256 rows; the others leave.  No workgroup ever waits for another, so
//      nothing depends on which workgroups are resident together and the
//      kernel can share the device with any other work;
//   3. the workgroup that completes the root holds, in the rows it selected,
//      the factored pivot block [L11 \ U11] (partial pivoting on original
//      rows); it writes the block, U11^-1, L11^-1 (for the block-row solve),
//      the reference's sequential swap list ipiv[k + j] and the list of rows
//      that the swaps move.
// k_tslu_apply, one workgroup per 64 panel rows: L21 = A21 U11^-1 on the
//   matrix cores for the rows that are not pivots, each written to its final
//   position; the first workgroup writes the pivot block to rows k..k+w-1.
#include <climits>

#include "kernels.hpp"
#include "mfma.hpp"
#include "wave.hpp"

namespace rlg {

constexpr int TW = 64;    // panel width
constexpr int TLR = 256;  // rows per leaf = threads per workgroup
constexpr int TF = 4;     // children per tree node: 4 x 64 candidates = 256 rows
constexpr int TG = 16;    // columns held in registers at a time
static_assert(TF * TW == TLR, "a merge has as many rows as a leaf");

// Tree of L leaves: level 0 has L nodes, level l + 1 has ceil(n_l / TF).
static size_t tree_nodes(size_t leaves) {
    size_t tot = 0, c = leaves;
    for (;;) {
        tot += c;
        if (c == 1) return tot;
        c = (c + TF - 1) / TF;
    }
}

struct TsluWork {
    int *cand;        // [nodes][TW] row numbers of a node's winners (-1: none)
    unsigned *cnt;    // [nodes] arrival counts, zero between panels
    float *F;         // [TW][TW] factored pivot block, row j = pivot j
    float *Uinv;      // [TW][TW] U11^-1, zero outside w x w
    int *sel;         // [TW] pivot rows in order
    int *map;         // [1 + 2 TW]: count, then (source row, destination) pairs
    int leaves_max;
};

static size_t al(size_t x) { return (x + 255) & ~(size_t)255; }

static size_t leaves_for(size_t rows) { return (rows + TLR - 1) / TLR; }

size_t tslu_work_bytes(size_t n) {
    const size_t nodes = tree_nodes(leaves_for(n ? n : 1));
    return al(nodes * TW * 4) + al(nodes * 4) + 2 * al(TW * TW * 4) + al(TW * 4) + al((1 + 2 * TW) * 4);
}

static TsluWork tslu_carve(void *work, size_t n) {
    const size_t nodes = tree_nodes(leaves_for(n ? n : 1));
    char *p = static_cast<char *>(work);
    TsluWork t;
    t.cand = reinterpret_cast<int *>(p); p += al(nodes * TW * 4);
    t.cnt = reinterpret_cast<unsigned *>(p); p += al(nodes * 4);
    t.F = reinterpret_cast<float *>(p); p += al(TW * TW * 4);
    t.Uinv = reinterpret_cast<float *>(p); p += al(TW * TW * 4);
    t.sel = reinterpret_cast<int *>(p); p += al(TW * 4);
    t.map = reinterpret_cast<int *>(p);
    t.leaves_max = (int)leaves_for(n ? n : 1);
    return t;
}

int tslu_reset(hipStream_t s, void *work, size_t n) {
    const size_t nodes = tree_nodes(leaves_for(n ? n : 1));
    return fill_u32(tslu_carve(work, n).cnt, nodes, 0u, s);
}

// Shared memory of the tournament kernel (69 KB, so that one workgroup fits
// beside one of the look-ahead's update): the 256 x 64 tile and the
// partial-pivoting state, and at the root, in the tile's place, the pivot block
// and the two triangles being inverted.
struct TourneyShared {
    union {
        float tile[TLR * TW];      // see `at`
        struct {
            float F[TW][TW + 1];
            float L[TW][TW + 1];   // L11, then L11^-1
            float Ut[TW][TW + 1];  // U11^T, then (U11^-1)^T
            float tmp[2][32][33];
        };
    };
    float u[TG][TW - TG];          // U12 of a group of columns
    unsigned long long act[4];     // rows of the tile not yet chosen
    int id[TLR];                   // row numbers (-1: none)
    int slot[TW];                  // tile row of pivot j (-1: not known yet, -2: none)
    int order[TW];                 // its row number
    int s_last;
};

// Entry (row, col) of the tile.  The 16-byte pieces of a row are permuted by its
// number, so that 16 consecutive rows read at one column touch all banks.
__device__ __forceinline__ int at(int row, int col) {
    return row * TW + (((col >> 2) ^ (row & 15)) << 2) + (col & 3);
}

// Rows sh.id[] of the panel into the tile (columns k .. k+w-1, zeros beyond).
__device__ __forceinline__ void load_rows(TourneyShared &sh, const float *__restrict__ A, long lda, int k, int w,
                                          bool vec) {
    const int tid = opaque(threadIdx.x), c = (tid & 15) * 4, r0 = tid >> 4;
    float4 v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int id = sh.id[q * 16 + r0];
        const float *r = A + (long)id * lda + k + c;
        v[q] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (id < 0) continue;
        if (vec && w == TW) {
            v[q] = *reinterpret_cast<const float4 *>(r);
        } else {
            if (c < w) v[q].x = r[0];
            if (c + 1 < w) v[q].y = r[1];
            if (c + 2 < w) v[q].z = r[2];
            if (c + 3 < w) v[q].w = r[3];
        }
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) *reinterpret_cast<float4 *>(&sh.tile[at(q * 16 + r0, c)]) = v[q];
}

__device__ __forceinline__ void publish_slot(TourneyShared &sh, int i, int t) {
    if ((threadIdx.x & 63) == 0)
        __hip_atomic_store(&sh.slot[i], t, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Columns cb .. cb+15 of the tile, by one wave: lane l holds rows l, l + 64, l + 128 and l + 192 in registers, so that a
// column needs no barrier.  The pivot is the largest |value| of the rows not yet
// chosen (ties: any; the choice is free for the tournament).  Every lane sets
// its best row's entries aside while the maximum is found, so that no branch
// (about 120 cycles) follows it; the winner's reach all lanes through scalar
// registers, and the other rows form their multipliers and are eliminated.
// Every column goes to the tile as it is done, then its pivot's row to sh.slot.
__device__ __forceinline__ void factor_group(TourneyShared &sh, int cb, int w) {
    const int lane = opaque(threadIdx.x & 63);
    float x[4][TG];
    unsigned long long act[4];  // rows not yet chosen
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        act[r] = uniform(sh.act[r]);
#pragma unroll
        for (int q = 0; q < TG; q += 4) {
            const float4 v = *reinterpret_cast<const float4 *>(&sh.tile[at(r * 64 + lane, cb + q)]);
            x[r][q] = v.x; x[r][q + 1] = v.y; x[r][q + 2] = v.z; x[r][q + 3] = v.w;
        }
    }
    int prev = -2;                // the pivot before: its tile row (-2: none)
    float m[4] = {}, u[TG] = {};  // of the pivot before: its elimination is completed
    unsigned key[4];              // while the next maximum is found
#pragma unroll
    for (int r = 0; r < 4; ++r) key[r] = bit_of(act[r], (__float_as_uint(x[r][0]) << 1) | 1u, 0u);
    static_for<TG>([&](auto cc) __attribute__((always_inline)) {
        constexpr int c = decltype(cc)::value;
        constexpr int N = c > 0 ? 4 * (TG - 1 - c) : 0;  // multiply-adds left of the pivot before
        auto eliminate = [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
#pragma unroll
            for (int f = i * N / 6; f < (i + 1) * N / 6; ++f)
                x[f % 4][c + 1 + f / 4] = fmaf(-m[f % 4], u[c + 1 + f / 4], x[f % 4][c + 1 + f / 4]);
            __builtin_amdgcn_sched_barrier(0);
        };
        const bool up0 = key[1] > key[0], up1 = key[3] > key[2];
        const unsigned k0 = max(key[0], key[1]), k1 = max(key[2], key[3]);
        const bool up = k1 > k0;
        const unsigned kk = max(k0, k1);
        unsigned d = dpp_max<DPP_SHR<1>>(kk);
        eliminate(std::integral_constant<int, 0>{});
        d = dpp_max<DPP_SHR<2>>(d);
        eliminate(std::integral_constant<int, 1>{});
        d = dpp_max<DPP_SHR<4>>(d);
        eliminate(std::integral_constant<int, 2>{});
        d = dpp_max<DPP_SHR<8>>(d);
        eliminate(std::integral_constant<int, 3>{});
        d = dpp_max<DPP_BCAST15>(d);
        eliminate(std::integral_constant<int, 4>{});
        d = dpp_max<DPP_BCAST31>(d);
        eliminate(std::integral_constant<int, 5>{});
        const unsigned mx = lane_get(d, 63);
        const unsigned long long b0 = __ballot(up0), b1 = __ballot(up1), b2 = __ballot(up);
        float y[TG];
#pragma unroll
        for (int e = c; e < TG; ++e) {
            const float v0 = up0 ? x[1][e] : x[0][e], v1 = up1 ? x[3][e] : x[2][e];
            y[e] = up ? v1 : v0;
        }
        const int l = __builtin_ctzll(__ballot(kk == mx));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = c; e < TG; ++e) u[e] = lane_get(y[e], l);
        const unsigned long long one = 1ull << l;
        act[0] &= ~(one & ~b2 & ~b0);
        act[1] &= ~(one & ~b2 & b0);
        act[2] &= ~(one & b2 & ~b1);
        act[3] &= ~(one & b2 & b1);
        const float rp = u[c] != 0.f ? __builtin_amdgcn_rcpf(u[c]) : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // a chosen row keeps its values: its multiplier is zero
            m[r] = bit_of(act[r], x[r][c] * rp, 0.f);
            if constexpr (c + 1 < TG) {
                x[r][c + 1] = fmaf(-m[r], u[c + 1], x[r][c + 1]);
                key[r] = bit_of(act[r], (__float_as_uint(x[r][c + 1]) << 1) | 1u, 0u);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // (the columns before are in the tile by now: the release does not wait)
        if constexpr (c > 0) publish_slot(sh, cb + c - 1, prev);
        const int o = (int)((b2 >> l) & 1), in = (int)((o ? b1 >> l : b0 >> l) & 1);
        const int t = (2 * o + in) * 64 + l;
        prev = mx != 0u && cb + c < w ? t : -2;  // (0: no row was left)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            x[r][c] = bit_of(act[r], m[r], x[r][c]);
            sh.tile[at(r * 64 + lane, cb + c)] = x[r][c];
        }
    });
    publish_slot(sh, cb + TG - 1, prev);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) sh.act[r] = act[r];
    }
}

// The pivot rows' part right of columns cb .. cb+15 (cb < 48), U12 = L11^-1 A12,
// one column per lane: by another wave behind factor_group, a row as soon as its
// pivot is known.  factor_group waits for nothing, so the wait ends; it is bounded
// all the same.
__device__ __forceinline__ void solve_group(TourneyShared &sh, int cb) {
    const int lane = opaque(threadIdx.x & 63);
    const int rest = TW - TG - cb, col = min(cb + TG + lane, TW - 1);
    float u12[TG];
    static_for<TG>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        int t = -1;
        for (int spin = 0; t == -1 && spin < (1 << 20); ++spin) {
            t = __hip_atomic_load(&sh.slot[cb + i], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (t == -1) __builtin_amdgcn_s_sleep(1);
        }
        t = __builtin_amdgcn_readfirstlane(t);
        const int r = max(t, 0);
        float l[TG], v = sh.tile[at(r, col)];
#pragma unroll
        for (int q = 0; q < i; ++q) l[q] = sh.tile[at(r, cb + q)];
#pragma unroll
        for (int q = 0; q < i; ++q) v = fmaf(-l[q], u12[q], v);
        u12[i] = v;
        if (lane < rest) {
            sh.u[i][lane] = v;
            if (i && t >= 0) sh.tile[at(r, col)] = v;
        }
    });
}

// Partial pivoting on the 256 rows of the tile, 16 columns at a time: wave 0
// factors them, wave 1 solves the pivot rows' part right of them meanwhile, then
// all waves update the other rows on the matrix cores.  On return the row chosen
// at step j (sh.slot, sh.order) holds its multipliers left of column j and its U
// row from column j on.
//
// Bound by the serial chain per column, about 115 instructions of one wave (a
// lone wave issues one in 4.3 to 6 cycles).  One row per thread, with the search
// and the pivot row going through LDS and a barrier per column, took 250 us for a
// panel on average over a factorization of order 16384 (four levels at most,
// beside the trailing update); this form takes 142, and a level on an idle device
// 32 instead of 58.  Branching to the winner's row instead of setting the best
// entries aside takes as long; with the solve in the same wave, 147.
__device__ void gepp256(TourneyShared &sh, int w) {
    using Acc = Mfma<float>::acc;
    const int wave = threadIdx.x >> 6;
#pragma unroll 1
    for (int cb = 0; cb < w; cb += TG) {
        const int lane = opaque(threadIdx.x & 63), lr = lane & 15, lk = lane >> 4;
        if (wave == 0) {
            __builtin_amdgcn_s_setprio(3);  // ahead of another kernel's waves on this SIMD
            factor_group(sh, cb, w);
            __builtin_amdgcn_s_setprio(0);
        } else if (wave == 1 && cb + TG < w) {
            __builtin_amdgcn_s_setprio(3);
            solve_group(sh, cb);
            __builtin_amdgcn_s_setprio(0);
        }
        __syncthreads();
        if (cb + TG >= w) break;
        // this wave's 64 rows: A22 -= L21 U12, the sums of 16 products kept
        // apart; chosen rows keep their values (their multipliers count as zero)
        float af[4][4];
        const unsigned long long act = sh.act[wave];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const float v = sh.tile[at(wave * 64 + rt * 16 + lr, cb + 4 * s + lk)];
                af[rt][s] = (act >> (rt * 16 + lr)) & 1ull ? v : 0.f;
            }
#pragma unroll 1
        for (int ct = cb + TG; ct < TW; ct += 16) {
            float bf[4], cv[4][4];
#pragma unroll
            for (int s = 0; s < 4; ++s) bf[s] = sh.u[4 * s + lk][ct - cb - TG + lr];
#pragma unroll
            for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r) cv[rt][r] = sh.tile[at(wave * 64 + rt * 16 + Mfma<float>::row(lk, r), ct + lr)];
            Acc acc[4] = {};
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int rt = 0; rt < 4; ++rt) acc[rt] = Mfma<float>::op(af[rt][s], bf[s], acc[rt]);
#pragma unroll
            for (int rt = 0; rt < 4; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    sh.tile[at(wave * 64 + rt * 16 + Mfma<float>::row(lk, r), ct + lr)] = cv[rt][r] - acc[rt][r];
        }
        __syncthreads();
    }
    const int tid = threadIdx.x;
    if (tid < TW) {
        const int t = sh.slot[tid];
        sh.order[tid] = t >= 0 ? sh.id[t] : -1;
    }
    __syncthreads();
}

// In-place inverses of two lower-triangular 64 x 64 matrices, M0 with a unit
// diagonal and M1 with its own (the upper parts are zero and stay zero).  The
// eight 16 x 16 diagonal blocks first, two per wave, a lane forward-substituting
// one column of the identity in registers; then the blocks below them,
// X21 = -X22 (M21 X11), by halves of 16 and of 32 on the matrix cores.  `tmp` is
// scratch.  Called by the whole workgroup.
//
// Bound by the substitutions' chains: 32 x 32 blocks took 15,500 cycles, these
// take 8,400.
__device__ void inv_lower64_pair(float (*M0)[TW + 1], float (*M1)[TW + 1], float (*tmp)[32][33]) {
    using Acc = Mfma<float>::acc;
    constexpr int B = 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    float (*const Mw)[TW + 1] = wave < 2 ? M0 : M1;
    if (lane < 2 * B) {
        const bool unit = wave < 2;
        const int o = ((wave & 1) * 2 + (lane >> 4)) * B, j = lane & 15;
        float x[B];
#pragma unroll
        for (int i = 0; i < B; ++i) {
            float s = (i == j) ? 1.f : 0.f;
#pragma unroll
            for (int q = 0; q < i; ++q) s -= Mw[o + i][o + q] * x[q];
            x[i] = unit ? s : s / Mw[o + i][o + i];
        }
        // every read of the block precedes the wave's writes to it
#pragma unroll
        for (int i = 0; i < B; ++i) Mw[o + i][o + j] = x[i];
    }
    __syncthreads();
    {   // the 32 x 32 half at o of this wave's matrix
        const int o = (wave & 1) * 2 * B;
        Acc acc = Acc{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < B / 4; ++s)
            acc = Mfma<float>::op(Mw[o + B + lr][o + 4 * s + lk], Mw[o + 4 * s + lk][o + lr], acc);
        float (*const t)[33] = &tmp[wave >> 1][(wave & 1) * B];
#pragma unroll
        for (int r = 0; r < 4; ++r) t[Mfma<float>::row(lk, r)][lr] = acc[r];
        __syncthreads();
        acc = Acc{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < B / 4; ++s)
            acc = Mfma<float>::op(Mw[o + B + lr][o + B + 4 * s + lk], t[4 * s + lk][lr], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) Mw[o + B + Mfma<float>::row(lk, r)][o + lr] = -acc[r];
    }
    __syncthreads();
    constexpr int H = TW / 2;
    const int tr = (wave >> 1) * 16, tc = (wave & 1) * 16;
#pragma unroll
    for (int q = 0; q < 2; ++q) {   // tmp = M21 X11
        float (*M)[TW + 1] = q ? M1 : M0;
        Acc acc = Acc{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < H / 4; ++s) acc = Mfma<float>::op(M[H + tr + lr][4 * s + lk], M[4 * s + lk][tc + lr], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) tmp[q][tr + Mfma<float>::row(lk, r)][tc + lr] = acc[r];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q) {   // X21 = -X22 tmp, over M21
        float (*M)[TW + 1] = q ? M1 : M0;
        Acc acc = Acc{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < H / 4; ++s)
            acc = Mfma<float>::op(M[H + tr + lr][H + 4 * s + lk], tmp[q][4 * s + lk][tc + lr], acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) M[H + tr + Mfma<float>::row(lk, r)][tc + lr] = -acc[r];
    }
    __syncthreads();
}

__global__ __launch_bounds__(TLR) __attribute__((amdgpu_waves_per_eu(2))) void k_tslu_tourney(const float *__restrict__ A, long lda, int k, int m,
                                                      int w, int64_t *__restrict__ ipiv,
                                                      int64_t *__restrict__ info, int n,
                                                      float *__restrict__ linv, TsluWork tw, int vec) {
    __shared__ __attribute__((aligned(16))) TourneyShared sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r0 = blockIdx.x * TLR;
    int id = r0 + tid < m ? k + r0 + tid : -1;  // the leaf's rows
    int level_off = 0, level_n = gridDim.x, node = blockIdx.x;
    for (;;) {
        sh.id[tid] = id;
        const unsigned long long have = __ballot(id >= 0);
        if (lane == 0) sh.act[wave] = have;
        if (tid < TW) sh.slot[tid] = -1;
        __syncthreads();
        load_rows(sh, A, lda, k, w, vec != 0);
        __syncthreads();
        gepp256(sh, w);
        if (level_n == 1) break;
        if (tid < TW) tw.cand[(level_off + node) * TW + tid] = sh.order[tid];

        // ---- the workgroup completing a node's last child merges it
        const int parent = node / TF;
        const int next_off = level_off + level_n, next_n = (level_n + TF - 1) / TF;
        const int kids = min(TF, level_n - parent * TF);
        __threadfence();  // this workgroup's winners before its arrival
        __syncthreads();
        if (tid == 0) {
            unsigned *c = &tw.cnt[next_off + parent];
            const unsigned old = atomicAdd(c, 1u);
            sh.s_last = old == (unsigned)(kids - 1);
            if (sh.s_last) *c = 0u;  // every child has arrived: ready for the next panel
        }
        __syncthreads();
        if (!sh.s_last) return;
        __threadfence();  // the other children's winners after their arrivals
        const int child = parent * TF + tid / TW;
        id = tid / TW < kids ? __hip_atomic_load(&tw.cand[(level_off + child) * TW + (tid % TW)],
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                             : -1;
        level_off = next_off;
        level_n = next_n;
        node = parent;
    }

    // ---- root: the pivot block, its inverses, the swaps
    {
        constexpr int PER = TW * TW / TLR;
        float f[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int r = q * 4 + wave, t = sh.slot[r];
            f[q] = t >= 0 ? sh.tile[at(t, lane)] : (r == lane && r >= w ? 1.f : 0.f);
        }
        __syncthreads();  // the tile has been read
        // L11 (unit lower) and U11^T, zero-padded to 64 x 64 with unit diagonal
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int r = q * 4 + wave, c = lane;
            sh.F[r][c] = f[q];
            sh.L[r][c] = c < r ? (r < w && c < w ? f[q] : 0.f) : 0.f;
            sh.Ut[c][r] = c >= r ? (r < w && c < w ? f[q] : (r == c ? 1.f : 0.f)) : 0.f;
            tw.F[r * TW + c] = f[q];
        }
    }
    __syncthreads();
    inv_lower64_pair(sh.L, sh.Ut, sh.tmp);
    for (int e = tid; e < TW * TW; e += TLR) {
        const int r = e / TW, c = e % TW;
        const bool in = r < w && c < w;
        linv[e] = in && c <= r ? sh.L[r][c] : 0.f;
        tw.Uinv[e] = in && c >= r ? sh.Ut[c][r] : 0.f;
    }
    if (wave == 0) {
        // The reference's sequential swaps: step j exchanges position k + j with
        // the position that holds pivot j's row now, to(j).  A row outside the top
        // w positions stays until it is chosen; one at top position q < j has gone
        // to to(q) by step j, and on from there if that is a top position below j.
        // Step j moves what position k + j holds then: what the last earlier step
        // that named that position brought there, or row k + j.
        const bool has = lane < w;
        const int selj = has ? sh.order[lane] : -1;
        if (has) tw.sel[lane] = selj;
        // (a pivot without a row cannot occur when m >= w; it would leave its
        // step without a swap, and info reports it)
        int to = selj < 0 ? k + lane : selj;
        for (unsigned long long open; (open = __ballot(has && to < k + lane)) != 0;) {
            const int q = max(to - k, 0) & 63;
            const int next = __builtin_amdgcn_ds_bpermute(q * 4, to);
            if (((open >> lane) & 1ull) && !((open >> q) & 1ull)) to = next;
        }
        sh.slot[lane] = -1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        if (has && to > k + lane && to < k + w) atomicMax(&sh.slot[to - k], lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        int held = lane;  // the top row that position k + lane holds at step `lane`
        const int before = sh.slot[lane];
        for (int go = before; __ballot(go >= 0) != 0;) {
            held = go >= 0 ? go : held;
            const int next = __builtin_amdgcn_ds_bpermute(held * 4, before);
            go = go >= 0 ? next : -1;
        }
        if (has) ipiv[k + lane] = to;
        // a top row that is a pivot itself does not stay where it was moved to
        sh.slot[lane] = 0;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        if (selj >= k && selj < k + w) sh.slot[selj - k] = 1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        const int from = has && to >= k + w && !sh.slot[held] ? k + held : -1;
        // rows that end outside the top: the displaced rows
        const bool mv = from >= 0;
        const unsigned long long bm = __ballot(mv);
        const int ord = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bm >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((unsigned)bm, 0));
        if (mv) { tw.map[1 + 2 * ord] = from; tw.map[2 + 2 * ord] = to; }
        if (lane == 0) tw.map[0] = __popcll(bm);
        const bool bad = lane < w && (selj < 0 || !(fabsf(sh.F[lane][lane]) >= 1.1920929e-7f));
        const unsigned long long first = __ballot(bad);
        if (lane == 0 && first && *info == (int64_t)n) *info = k + __builtin_ctzll(first);
    }
}

// L21 = A21 U11^-1 for panel rows [k + 64 b, k + 64 b + 64), each written to
// its final position; the pivot rows are skipped (their factored rows come
// from the pivot block, which workgroup 0 writes over rows k .. k+w-1 after
// reading its own rows).  The destinations of moved rows are positions of
// pivot rows, whose original values no workgroup needs, so the in-place
// writes cannot race with another workgroup's reads.
__global__ __launch_bounds__(256) void k_tslu_apply(float *__restrict__ A, long lda, int k, int m, int w,
                                                    TsluWork tw) {
    using Acc = Mfma<float>::acc;
    __shared__ float Ui[TW][TW + 1];
    __shared__ float X[64][TW + 1];
    __shared__ int dst[64];
    __shared__ unsigned long long selmask;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lk = lane >> 4;
    const int base = k + (int)blockIdx.x * 64;
    const int rows = min(64, k + m - base);
    // every read is issued first: one memory latency, not one per phase (8.6 us a
    // launch on average at order 16384; with the lists and F read where they are
    // used, 11.6)
    constexpr int PER = 64 * TW / 256;
    const int chosen = tid < w ? tw.sel[tid] : -1;
    const int cnt = tw.map[0];  // at most 64
    const int from = tid < 64 ? tw.map[1 + 2 * tid] : -1, to = tid < 64 ? tw.map[2 + 2 * tid] : -1;
    float vf[PER];
    {
        float vu[PER], vx[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = q * 256 + tid, r = e / TW, c = e % TW;
            vu[q] = tw.Uinv[e];
            vx[q] = (r < rows && c < w) ? A[(long)(base + r) * lda + k + c] : 0.f;
        }
        if (blockIdx.x == 0) {
#pragma unroll
            for (int q = 0; q < PER; ++q) vf[q] = tw.F[q * 256 + tid];
        }
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = q * 256 + tid, r = e / TW, c = e % TW;
            Ui[r][c] = vu[q];
            X[r][c] = vx[q];
        }
    }
    if (tid < 64) dst[tid] = base + tid;
    if (tid == 0) selmask = 0ull;
    __syncthreads();
    if (chosen >= base && chosen < base + 64) atomicOr(&selmask, 1ull << (chosen - base));
    if (tid < cnt && from >= base && from < base + 64) dst[from - base] = to;
    __syncthreads();
    Acc acc[4];
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) acc[jc] = Acc{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < TW / 4; ++s) {
        const float av = X[16 * wave + lr][4 * s + lk];
#pragma unroll
        for (int jc = 0; jc < 4; ++jc) acc[jc] = Mfma<float>::op(av, Ui[4 * s + lk][16 * jc + lr], acc[jc]);
    }
    const unsigned long long sm = selmask;
#pragma unroll
    for (int jc = 0; jc < 4; ++jc)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * wave + Mfma<float>::row(lk, r), col = 16 * jc + lr;
            if (row < rows && col < w && !((sm >> row) & 1ull))
                A[(long)dst[row] * lda + k + col] = acc[jc][r];
        }
    if (blockIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = q * 256 + tid, r = e / TW, c = e % TW;
            if (r < w && c < w) A[(long)(k + r) * lda + k + c] = vf[q];
        }
    }
}

size_t tslu_max_rows(size_t n) { return leaves_for(n ? n : 1) * TLR; }

int tslu_panel(hipStream_t s, float *a, size_t lda, size_t k, size_t m, size_t w, int64_t *ipiv,
               int64_t *info, size_t n, void *work, float *linv) {
    const TsluWork tw = tslu_carve(work, n);
    const size_t L = leaves_for(m);
    if (L > (size_t)tw.leaves_max || w > (size_t)TW || w == 0 || m < w) {
        set_error("TSLU panel of %zu x %zu is out of range", m, w);
        return RLG_E_INVALID_ARG;
    }
    // row loads are 16-byte vectors when every panel row starts 16-byte aligned
    const int vec = (lda % 4 == 0 && k % 4 == 0 && ((uintptr_t)a & 15) == 0) ? 1 : 0;
    {
        // algorithmic bytes: the m x w panel read once (the leaves)
        RLG_PROF_W("tslu_tourney", s, (double)m * (double)w * 4.0);
        hipLaunchKernelGGL(k_tslu_tourney, dim3((unsigned)L), dim3(TLR), 0, s, a, (long)lda, (int)k, (int)m,
                           (int)w, ipiv, info, (int)n, linv, tw, vec);
        RLG_LAUNCHED();
    }
    {
        // algorithmic bytes: the panel read and written once
        RLG_PROF_W("tslu_apply", s, 2.0 * (double)m * (double)w * 4.0);
        hipLaunchKernelGGL(k_tslu_apply, dim3(ceil_div(m, 64)), dim3(256), 0, s, a, (long)lda, (int)k,
                           (int)m, (int)w, tw);
        RLG_LAUNCHED();
    }
    return RLG_OK;
}

}  // namespace rlg
