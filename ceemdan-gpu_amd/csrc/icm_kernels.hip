// HIP kernels of the ICEEMDAN hot path (gfx950, wave64).
//
// A knot set is stored as bitmasks: 64-bit words, one per 64 samples of a
// 256-sample tile and knot type, written by the kernel that wrote the
// samples; a knot's position is its bit, its value the sample there.  One
// sift pass of every series is three launches:
//   k_solve         one wavefront per window of 64*B knots: positions from
//                   the bitmasks, values from the samples, natural-spline
//                   rows, per-lane elimination of B rows, parallel cyclic
//                   reduction across the 64 lanes, back substitution -> c
//   k_sift_w        one wavefront per segment of tiles: interval of every
//                   sample from the tile's bitmasks, interval coefficients in
//                   LDS, upper/lower envelope, mean, subtract; then the
//                   extrema of the new samples as the next pass's bitmasks
//   k_knot_prefix_* per series: tile knot prefixes, neighbour knots of every
//                   tile, the solve's window list, the count of tiles too
//                   full for the small knot table
// From the second stage of a phase on, k_sift_w runs with a small knot table
// (more waves per SIMD) and k_sift_list sifts, with the full table, the tiles
// it could not hold (or every segment, when the count says they are many).
// Reference counterparts: find_extrema_shfl_* :92-148, CUB ExclusiveSum
// :859-883, select_extrema_* :150-207, setBoundary* :209-291,
// tridiagonal_setup :310-343, gtsv2_nopivot :899-921, spline_coefficients
// :382-401, interpolate :403-439, averageUppperLower :441-454,
// produceSX/thresholdJudge :456-492, updateRealizations :527-544
// (all cudaICEEMDAN.cu).
#include "icm_device.h"
#include "icm_kernels.h"
#include "icm_spline.h"

#include <map>
#include <mutex>
#include <type_traits>
#include <utility>
#include "icm_errors.h"

namespace icm {

// ------------------------------------------------------------ tile helpers

constexpr int kWKC = kWT / 2 + 8;      // table entries per type (>= cnt + 3 for any tile)
constexpr int kWKS = kWave;             // small table (sparse passes): tiles with cnt + 3 <= 64

// ------------------------------------------------------------- knot bitmasks
// A tile's knots of one type are the set bits of four 64-bit row masks
// m[r] (bit b of row r = sample 64 r + b of the tile).

// tile offset of the last set bit, -1 if none
__device__ __forceinline__ int mask_last(const uint64_t (&m)[kWR])
{
    int last = -1;
#pragma unroll
    for (int r = 0; r < kWR; ++r) last = m[r] ? kWave * r + 63 - __clzll(m[r]) : last;
    return last;
}

// Strict maxima and minima among one row of 64 samples from the row's
// comparisons with the sample after each (gt: v[p] > v[p + 1], lt: <) and
// the same two of the sample before the row (cg, cl: bit 0).  One comparison
// of neighbours serves both: v[p] > v[p - 1] is lt of p - 1, a scalar shift,
// so a row takes two compares and one neighbour row instead of four and two.
// Each comparison is balloted
// on its own: the ballot of a combination of flags costs a v_cndmask and a
// v_cmp.  The empty asm statement makes the two row masks scalar registers at
// this point (held together, the comparison masks of all rows spilled).
__device__ __forceinline__ void row_extrema(uint64_t gt, uint64_t lt, uint64_t& cg, uint64_t& cl,
                                            uint64_t& mx, uint64_t& mn)
{
    mx = gt & ((lt << 1) | cl);
    mn = lt & ((gt << 1) | cg);
    cg = gt >> 63;
    cl = lt >> 63;
    asm volatile("" : "+s"(mx), "+s"(mn));
}

// masks of the samples of row p0 .. p0 + 63 inside a series of N samples, and
// of its two ends (ends are knots of both types)
__device__ __forceinline__ void row_ends(int p0, int N, uint64_t& valid, uint64_t& end)
{
    const int left = N - p0;
    valid = left >= 64 ? ~0ull : left <= 0 ? 0ull : (1ull << left) - 1;
    end = p0 == 0 ? 1ull : 0ull;
    if (left >= 1 && left <= 64) end |= 1ull << (left - 1);
}

// tile offset of the first set bit, -1 if none
__device__ __forceinline__ int mask_first(const uint64_t (&m)[kWR])
{
    int first = -1;
#pragma unroll
    for (int r = kWR - 1; r >= 0; --r) first = m[r] ? kWave * r + __ffsll((long long)m[r]) - 1 : first;
    return first;
}

template <typename real>
__device__ __forceinline__ void load_masks(const KnotsDev<real>& k, int64_t gt, int type,
                                           uint64_t (&m)[kWR])
{
#pragma unroll
    for (int r = 0; r < kWR; ++r) m[r] = k.mask[8 * gt + kWR * type + r];
}

// The last knot and the one before it among some tiles (positions, -1 =
// none).  Positions are distinct, so combining two sets needs no order.
struct LastTwo {
    int a, b;
};

__device__ __forceinline__ LastTwo lt_combine(const LastTwo& A, const LastTwo& B)
{
    return LastTwo{max(A.a, B.a), max(max(A.b, B.b), min(A.a, B.a))};
}

__device__ __forceinline__ LastTwo lt_none() { return LastTwo{-1, -1}; }

// Inclusive scans over the lanes by lane moves inside the vector unit (two to
// five instructions a step; by ds_bpermute each took a round trip to LDS, and
// a decomposition of 16 ragged FP32 series x 100 took 177.2 ms instead of
// 174.7): sums, last two knots, and (downwards) the least value of the lanes
// from this one.
__device__ __forceinline__ int sum_scan(int v)
{
    v += dpp_row_i<0x111, 0xF>(v, 0);
    v += dpp_row_i<0x112, 0xF>(v, 0);
    v += dpp_row_i<0x114, 0xF>(v, 0);
    v += dpp_row_i<0x118, 0xF>(v, 0);
    v += dpp_row_i<0x142, 0xA>(v, 0);
    v += dpp_row_i<0x143, 0xC>(v, 0);
    return v;
}
template <int CTRL, int ROWS>
__device__ __forceinline__ void lt_step(LastTwo& v)
{
    v = lt_combine(LastTwo{dpp_row_i<CTRL, ROWS>(v.a, -1), dpp_row_i<CTRL, ROWS>(v.b, -1)}, v);
}
__device__ __forceinline__ LastTwo lt_scan(LastTwo v)
{
    lt_step<0x111, 0xF>(v);
    lt_step<0x112, 0xF>(v);
    lt_step<0x114, 0xF>(v);
    lt_step<0x118, 0xF>(v);
    lt_step<0x142, 0xA>(v);
    lt_step<0x143, 0xC>(v);
    return v;
}
__device__ __forceinline__ int suffix_min(int v)
{
    constexpr int INF = 0x7FFFFFFF;
    v = min(v, dpp_row_i<0x101, 0xF>(v, INF));
    v = min(v, dpp_row_i<0x102, 0xF>(v, INF));
    v = min(v, dpp_row_i<0x104, 0xF>(v, INF));
    v = min(v, dpp_row_i<0x108, 0xF>(v, INF));
    // rows 1, 2, 3 begin at lanes 16, 32, 48
    const int r3 = __builtin_amdgcn_readlane(v, 48), r2 = min(__builtin_amdgcn_readlane(v, 32), r3);
    const int r1 = min(__builtin_amdgcn_readlane(v, 16), r2);
    const int row = (threadIdx.x & 63) >> 4;
    return min(v, row == 0 ? r1 : row == 1 ? r2 : row == 2 ? r3 : INF);
}
// what the lanes before this one hold together (after a scan)
__device__ __forceinline__ LastTwo lt_before(const LastTwo& v) { return LastTwo{dpp_prev_i(v.a, -1), dpp_prev_i(v.b, -1)}; }

// Knot prefix: per-series exclusive scan of the tile knot counts (the CUB
// ExclusiveSum of cudaICEEMDAN.cu:859-883, over tiles instead of samples),
// the series knot counts, the solve's window items, and for every tile the
// positions and values of the two knots before it and of the first knot
// after it (positions from the bitmasks, values from the pass input h).
//
// The same outputs with one 1024-thread workgroup per series and one tile per
// thread (chunks of 1024 tiles): workgroup scans forward (counts, last two
// knots) and backward (next knot), carried from chunk to chunk.
constexpr int kPT = 1024;

// Window item w of a series with wmx windows of maxima and wmn of minima:
// the two types alternate (maxima window i, then minima window i), so the
// two windows over one stretch of samples go to neighbouring waves of one
// solve workgroup and read the same cache lines at about the same time.
__device__ __forceinline__ void window_of_item(int w, int wmx, int wmn, int& type, int& wi)
{
    const int m = min(wmx, wmn);
    if (w < 2 * m) {
        type = w & 1;
        wi = w >> 1;
    } else {
        type = wmx > wmn ? 0 : 1;
        wi = m + (w - 2 * m);
    }
}

template <typename real>
__global__ __launch_bounds__(kPT) void k_knot_prefix_b(SeriesDev sd, KnotsDev<real> k, const real* h,
                                                       PassCtl pc, const int* active)
{
    constexpr int NWV = kPT / kWave;
    constexpr int INF = 0x7FFFFFFF;
    __shared__ int s_tot[NWV], s_ex_tot[NWV], s_all;
    __shared__ LastTwo s_lt[NWV], s_ex_lt[NWV], s_all_lt;
    __shared__ int s_min[NWV];
    __shared__ unsigned s_wbase;
    const int s = blockIdx.x;
    if (pc.run && load_scalar(pc.run) == 0u) return;
    if (active && !active[s]) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int tb = sd.tile0[s], nt = sd.ntl[s];
    const real* hs = h + sd.off[s];
    {
        // tiles the small sift table cannot hold
        unsigned d = 0;
        for (int t = tid; t < nt; t += kPT) {
            const int c0 = k.cnt[2 * (tb + t)], c1 = k.cnt[2 * (tb + t) + 1];
            d += (c0 + 3 > kWKS || c1 + 3 > kWKS) ? 1u : 0u;
        }
        for (int o = 32; o >= 1; o >>= 1) d += __shfl_xor(d, o, kWave);
        if (lane == 0 && d) atomicAdd(&pc.dense[pc.epoch], d);
    }
    int ntot[2] = {0, 0};
    for (int ty = 0; ty < 2; ++ty) {
        // forward: exclusive count and the last two knots before each tile
        int carry = 0;
        LastTwo carry_lt = lt_none();
        for (int base = 0; base < nt; base += kPT) {
            const int t = base + tid;
            const int c = t < nt ? k.cnt[2 * (tb + t) + ty] : 0;
            LastTwo own = lt_none();
            if (c > 0) {
                uint64_t m[kWR];
                load_masks(k, tb + t, ty, m);
                const int b1 = mask_last(m);
                m[b1 / kWave] ^= 1ull << (b1 % kWave);
                own.a = t * kWT + b1;
                own.b = c >= 2 ? t * kWT + mask_last(m) : -1;
            }
            const int inc = sum_scan(c);
            const LastTwo sc = lt_scan(own);
            const int xi = dpp_prev_i(inc, 0);
            const LastTwo xl = lt_before(sc);
            __syncthreads();   // earlier readers of s_* are done
            if (lane == kWave - 1) {
                s_tot[wv] = inc;
                s_lt[wv] = sc;
            }
            __syncthreads();
            if (wv == 0) {
                // exclusive scan of the wave totals by the first NWV lanes
                const int v = lane < NWV ? s_tot[lane] : 0;
                const int vi = sum_scan(v);
                const LastTwo li = lt_scan(lane < NWV ? s_lt[lane] : lt_none());
                const LastTwo le = lt_before(li);
                if (lane < NWV) {
                    s_ex_tot[lane] = vi - v;
                    s_ex_lt[lane] = le;
                }
                if (lane == NWV - 1) {
                    s_all = vi;
                    s_all_lt = li;
                }
            }
            __syncthreads();
            const int ex = carry + s_ex_tot[wv] + xi;
            const LastTwo before = lt_combine(carry_lt, lt_combine(s_ex_lt[wv], xl));
            if (t < nt) {
                k.pre[2 * (tb + t) + ty] = ex;
                const int64_t o = 6 * (int64_t)(tb + t) + 3 * ty;
                k.nbx[o] = before.a;
                k.nby[o] = before.a >= 0 ? hs[before.a] : (real)0;
                k.nbx[o + 1] = before.b;
                k.nby[o + 1] = before.b >= 0 ? hs[before.b] : (real)0;
                if (k.left) k.left[2 * (tb + t) + ty] = before.a;
            }
            carry += s_all;
            carry_lt = lt_combine(carry_lt, s_all_lt);
        }
        ntot[ty] = carry;
        // backward: first non-empty tile after each tile
        int carry_min = INF;
        for (int base = ((nt - 1) / kPT) * kPT; base >= 0; base -= kPT) {
            const int t = base + tid;
            const int c = t < nt ? k.cnt[2 * (tb + t) + ty] : 0;
            const int mn = suffix_min(c > 0 ? t : INF);
            const int xm = dpp_next_i(mn, INF);
            __syncthreads();
            if (lane == 0) s_min[wv] = mn;
            __syncthreads();
            int after = min(carry_min, xm);
            int all = carry_min;
            for (int w = 0; w < NWV; ++w) {
                if (w > wv) after = min(after, s_min[w]);
                all = min(all, s_min[w]);
            }
            if (t < nt) {
                const int64_t o = 6 * (int64_t)(tb + t) + 3 * ty + 2;
                int x3 = -1;
                if (after != INF) {
                    uint64_t m[kWR];
                    load_masks(k, tb + after, ty, m);
                    x3 = after * kWT + mask_first(m);
                }
                k.nbx[o] = x3;
                k.nby[o] = x3 >= 0 ? hs[x3] : (real)0;
                if (k.right) k.right[2 * (tb + t) + ty] = x3;
            }
            carry_min = all;
        }
    }
    const int wmx = (ntot[0] + pc.K - 1) / pc.K;
    const int wmn = (ntot[1] + pc.K - 1) / pc.K;
    if (tid == 0) {
        k.n[2 * s] = ntot[0];
        k.n[2 * s + 1] = ntot[1];
        s_wbase = atomicAdd(pc.wincount, (unsigned)(wmx + wmn));
    }
    __syncthreads();
    const unsigned wbase = s_wbase;
    for (int w = tid; w < wmx + wmn; w += kPT) {
        int type, wi;
        window_of_item(w, wmx, wmn, type, wi);
        pc.winlist[kWinItem * (wbase + w)] = s;
        pc.winlist[kWinItem * (wbase + w) + 1] = (wi << 1) | type;
        pc.winlist[kWinItem * (wbase + w) + 2] = -1;   // no tile hint: the solve searches
    }
}

// Series of at most 1024 tiles: the same outputs in one pass, both knot
// types and both scan directions at once (one load round, two workgroup
// barriers, one gather round).
template <typename real>
__global__ __launch_bounds__(kPT) void k_knot_prefix_1(SeriesDev sd, KnotsDev<real> k, const real* h,
                                                       PassCtl pc, const int* active)
{
    constexpr int NWV = kPT / kWave;
    constexpr int INF = 0x7FFFFFFF;
    __shared__ int s_tot[2][NWV], s_ex_tot[2][NWV], s_all[2];
    __shared__ LastTwo s_lt[2][NWV], s_ex_lt[2][NWV];
    __shared__ int s_min[2][NWV], s_ex_min[2][NWV];
    __shared__ int s_pre[2][kPT];
    __shared__ int s_first[2][kPT];
    __shared__ unsigned s_wbase;
    __shared__ unsigned s_dense[NWV];
    const int s = blockIdx.x;
    if (pc.run && load_scalar(pc.run) == 0u) return;
    if (active && !active[s]) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int tb = sd.tile0[s], nt = sd.ntl[s];
    const real* hs = h + sd.off[s];
    const int t = tid;
    int c[2];
    LastTwo sc[2];
    int inc[2], mn[2];
    int first[2];         // tile offset of the tile's first knot per type
    // both types' counts, then both types' bitmasks, in one round trip each
    c[0] = t < nt ? k.cnt[2 * (tb + t)] : 0;
    c[1] = t < nt ? k.cnt[2 * (tb + t) + 1] : 0;
    // the bitmasks loaded with the counts (not after them, for the tiles
    // with knots only): one round trip fewer per workgroup
    uint64_t mm[2][kWR];
#pragma unroll
    for (int q = 0; q < 2 * kWR; ++q)
        mm[q / kWR][q % kWR] = t < nt ? k.mask[8 * (int64_t)(tb + min(t, nt - 1)) + q] : 0ull;
#pragma unroll
    for (int ty = 0; ty < 2; ++ty) {
        sc[ty] = lt_none();
        first[ty] = -1;
        if (c[ty] > 0) {
            uint64_t m[kWR];
#pragma unroll
            for (int r = 0; r < kWR; ++r) m[r] = mm[ty][r];
            first[ty] = mask_first(m);
            const int b1 = mask_last(m);
            m[b1 / kWave] ^= 1ull << (b1 % kWave);
            sc[ty].a = t * kWT + b1;
            sc[ty].b = c[ty] >= 2 ? t * kWT + mask_last(m) : -1;
        }
        inc[ty] = c[ty];
        mn[ty] = c[ty] > 0 ? t : INF;
    }
    {
        // tiles the small sift table cannot hold
        const unsigned d = (unsigned)__popcll(wave_ballot(c[0] + 3 > kWKS || c[1] + 3 > kWKS));
        if (lane == 0) s_dense[wv] = d;
    }
    int xi[2], xm[2];
    LastTwo xl[2];
#pragma unroll
    for (int ty = 0; ty < 2; ++ty) {
        inc[ty] = sum_scan(inc[ty]);
        sc[ty] = lt_scan(sc[ty]);
        mn[ty] = suffix_min(mn[ty]);
        xi[ty] = dpp_prev_i(inc[ty], 0);
        xl[ty] = lt_before(sc[ty]);
        xm[ty] = dpp_next_i(mn[ty], INF);
        if (lane == kWave - 1) {
            s_tot[ty][wv] = inc[ty];
            s_lt[ty][wv] = sc[ty];
        }
        if (lane == 0) s_min[ty][wv] = mn[ty];
        s_first[ty][t] = first[ty];
    }
    __syncthreads();
    if (wv == 0) {
        // scans of the wave totals by the first NWV lanes
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            const int v = lane < NWV ? s_tot[ty][lane] : 0;
            const int vi = sum_scan(v), mi = suffix_min(lane < NWV ? s_min[ty][lane] : INF);
            const LastTwo li = lt_scan(lane < NWV ? s_lt[ty][lane] : lt_none());
            const LastTwo le = lt_before(li);
            const int me = dpp_next_i(mi, INF);
            if (lane < NWV) {
                s_ex_tot[ty][lane] = vi - v;
                s_ex_lt[ty][lane] = le;
                s_ex_min[ty][lane] = me;
            }
            if (lane == NWV - 1) s_all[ty] = vi;
        }
    }
    __syncthreads();
    if (t < nt) {
        // positions of both types' neighbour knots, then all six value loads
        // (at clamped positions, so that none sits under a condition), then
        // the stores
        int ex[2], xs[2][3];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            ex[ty] = s_ex_tot[ty][wv] + xi[ty];
            const LastTwo before = lt_combine(s_ex_lt[ty][wv], xl[ty]);
            const int after = min(s_ex_min[ty][wv], xm[ty]);
            xs[ty][0] = before.a;
            xs[ty][1] = before.b;
            xs[ty][2] = after == INF ? -1 : after * kWT + s_first[ty][after];
        }
        real ys[2][3];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty)
#pragma unroll
            for (int w = 0; w < 3; ++w) ys[ty][w] = hs[max(xs[ty][w], 0)];
        if (tid == 0) {
            // the window base is requested while the values are in flight
            const int n0 = s_all[0], n1 = s_all[1];
            k.n[2 * s] = n0;
            k.n[2 * s + 1] = n1;
            s_wbase = atomicAdd(pc.wincount,
                                (unsigned)((n0 + pc.K - 1) / pc.K + (n1 + pc.K - 1) / pc.K));
        }
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            k.pre[2 * (tb + t) + ty] = ex[ty];
            s_pre[ty][t] = ex[ty];
            const int64_t o = 6 * (int64_t)(tb + t) + 3 * ty;
#pragma unroll
            for (int w = 0; w < 3; ++w) {
                k.nbx[o + w] = xs[ty][w];
                k.nby[o + w] = xs[ty][w] >= 0 ? ys[ty][w] : (real)0;
            }
            if (k.left) {
                k.left[2 * (tb + t) + ty] = xs[ty][0];
                k.right[2 * (tb + t) + ty] = xs[ty][2];
            }
        }
    }
    const int n0 = s_all[0], n1 = s_all[1];
    const int wmx = (n0 + pc.K - 1) / pc.K;
    const int wmn = (n1 + pc.K - 1) / pc.K;
    if (tid == 0 && nt == 0) {
        k.n[2 * s] = n0;
        k.n[2 * s + 1] = n1;
        s_wbase = atomicAdd(pc.wincount, (unsigned)(wmx + wmn));
    }
    if (tid == 0) {
        unsigned d = 0;
        for (int w = 0; w < NWV; ++w) d += s_dense[w];
        if (d) atomicAdd(&pc.dense[pc.epoch], d);
    }
    __syncthreads();
    const unsigned wbase = s_wbase;
    for (int w = tid; w < wmx + wmn; w += kPT) {
        int type, wi;
        window_of_item(w, wmx, wmn, type, wi);
        // the last tile whose knots start at or before the window's first
        // gathered knot, so the solve needs no search
        const int glo = max(wi * pc.K - pc.H - 1, 0);
        int x = 0, y = nt - 1;
        while (x < y) {
            const int mid = (x + y + 1) >> 1;
            if (s_pre[type][mid] <= glo) x = mid;
            else y = mid - 1;
        }
        pc.winlist[kWinItem * (wbase + w)] = s;
        pc.winlist[kWinItem * (wbase + w) + 1] = (wi << 1) | type;
        pc.winlist[kWinItem * (wbase + w) + 2] = x;
    }
}

// Series of at most kPT tiles: the same outputs with one wavefront per
// series and no workgroup barrier.  Lane l owns tile 64 j + l of chunk j;
// the wave scans each chunk (counts, and the last two knots before each
// tile) and carries the totals to the next chunk, with the next chunk's
// counts and bitmasks in flight meanwhile; a backward sweep over the chunks
// (suffix minimum of the tiles' first knots) gives the first knot after each
// tile.  Each window's first tile is known from the scan (the tile holding
// the window's first gathered knot) and kept in LDS until the series' window
// count is known.  Workgroups are four independent waves, so beside another
// stream's sift the kernel runs in whatever wave slots that kernel leaves
// free (a 1024-thread workgroup needs 16 free slots on one CU at once, and
// then waited for the other stream's sift to drain: 3.5 ms per pass beside
// it against 0.5 ms alone).
// windows per type of a series of at most kPT tiles: <= 129 knots per tile
// and type, K >= 448 rows kept per window
constexpr int kPWin = (kPT * 129 + 447) / 448 + 1;
// series length (tiles) up to which the one-wave kernel is used (a wave takes
// 64 tiles at a time, one after the other: on 200 series of 954 tiles it more
// than doubled what a decomposition spends outside init, solve and sift, 10.0
// -> 21.9 ms; where a 1024-thread workgroup would be mostly idle it is ahead)
constexpr int kPWTiles = 128;

template <typename real>
__global__ __launch_bounds__(kThreads) void k_knot_prefix_w(SeriesDev sd, KnotsDev<real> k, const real* h,
                                                            PassCtl pc, const int* active)
{
    constexpr int NW = kThreads / kWave;
    constexpr int INF = 0x7FFFFFFF;
    __shared__ int s_hint[NW][2][kPWin];
    const int lane = threadIdx.x & 63, wv = wave_index();
    const int s = blockIdx.x * NW + wv;
    if (s >= sd.nseries) return;
    if (pc.run && load_scalar(pc.run) == 0u) return;
    if (active && !load_scalar(active + s)) return;
    const int tb = load_scalar(sd.tile0 + s), nt = load_scalar(sd.ntl + s);
    const real* hs = h + load_scalar(sd.off + s);
    const int K = pc.K, H = pc.H;
    const int nch = (nt + kWave - 1) / kWave;

    // counts and the eight row bitmasks of tile 64 ch + lane (zero past the series)
    auto load = [&](int ch, int (&c)[2], uint64_t (&m)[2 * kWR]) {
        const int t = ch * kWave + lane;
        const bool in = t < nt;
        const int64_t gt = tb + (in ? t : 0);
        c[0] = in ? k.cnt[2 * gt] : 0;
        c[1] = in ? k.cnt[2 * gt + 1] : 0;
#pragma unroll
        for (int q = 0; q < 2 * kWR; ++q) m[q] = in ? k.mask[8 * gt + q] : 0ull;
    };

    int carry[2] = {0, 0};
    LastTwo carry_lt[2] = {lt_none(), lt_none()};
    unsigned dense = 0;   // tiles the small sift table cannot hold
    int c[2], cn[2] = {0, 0};
    uint64_t m[2 * kWR], mn[2 * kWR] = {};
    load(0, c, m);
    for (int ch = 0; ch < nch; ++ch) {
        if (ch + 1 < nch) load(ch + 1, cn, mn);
        const int t = ch * kWave + lane;
        const bool in = t < nt;
        const int64_t gt = tb + t;
        dense += (unsigned)__popcll(wave_ballot(in && (c[0] + 3 > kWKS || c[1] + 3 > kWKS)));
        int ex[2], xb[2][2], fp[2];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            uint64_t mm[kWR];
#pragma unroll
            for (int r = 0; r < kWR; ++r) mm[r] = m[ty * kWR + r];
            LastTwo own = lt_none();
            fp[ty] = -1;
            if (c[ty] > 0) {
                fp[ty] = t * kWT + mask_first(mm);
                const int b1 = mask_last(mm);
                mm[b1 / kWave] ^= 1ull << (b1 % kWave);
                own.a = t * kWT + b1;
                own.b = c[ty] >= 2 ? t * kWT + mask_last(mm) : -1;
            }
            const int inc = sum_scan(c[ty]);
            const LastTwo sc = lt_scan(own);
            ex[ty] = carry[ty] + inc - c[ty];
            const LastTwo before = lt_combine(carry_lt[ty], lt_before(sc));
            xb[ty][0] = before.a;
            xb[ty][1] = before.b;
            // the window whose first gathered knot (max(w K - H - 1, 0)) lies
            // in this tile: at most one, as K exceeds a tile's knots
            if (c[ty] > 0) {
                if (ex[ty] == 0) s_hint[wv][ty][0] = t;
                const int w = (ex[ty] + c[ty] + H) / K;
                if (w >= 1 && w < kPWin && w * K - H - 1 >= ex[ty]) s_hint[wv][ty][w] = t;
            }
            carry[ty] += __builtin_amdgcn_readlane(inc, kWave - 1);
            carry_lt[ty] = lt_combine(carry_lt[ty], LastTwo{__builtin_amdgcn_readlane(sc.a, kWave - 1),
                                                            __builtin_amdgcn_readlane(sc.b, kWave - 1)});
        }
        // values of the knots before the tile (positions of knots that exist,
        // or 0), all loads before the stores
        real yb[2][2];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty)
#pragma unroll
            for (int w = 0; w < 2; ++w) yb[ty][w] = hs[max(xb[ty][w], 0)];
        if (in) {
#pragma unroll
            for (int ty = 0; ty < 2; ++ty) {
                k.pre[2 * gt + ty] = ex[ty];
                const int64_t o = 6 * gt + 3 * ty;
                k.nbx[o] = xb[ty][0];
                k.nby[o] = xb[ty][0] >= 0 ? yb[ty][0] : (real)0;
                k.nbx[o + 1] = xb[ty][1];
                k.nby[o + 1] = xb[ty][1] >= 0 ? yb[ty][1] : (real)0;
                // the tile's own first knot, read back by this lane below
                k.nbx[o + 2] = fp[ty];
                if (k.left) k.left[2 * gt + ty] = xb[ty][0];
            }
        }
        c[0] = cn[0];
        c[1] = cn[1];
#pragma unroll
        for (int q = 0; q < 2 * kWR; ++q) m[q] = mn[q];
    }
    // backward: the first knot after each tile = the least first knot of
    // the tiles after it
    int cmin[2] = {INF, INF};
    for (int ch = nch - 1; ch >= 0; --ch) {
        const int t = ch * kWave + lane;
        const bool in = t < nt;
        const int64_t gt = tb + (in ? t : 0);
        int after[2];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            const int f = in ? k.nbx[6 * gt + 3 * ty + 2] : -1;
            const int mnv = suffix_min(f >= 0 ? f : INF);
            after[ty] = min(cmin[ty], dpp_next_i(mnv, INF));
            cmin[ty] = min(cmin[ty], __builtin_amdgcn_readlane(mnv, 0));
        }
        real ya[2];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) ya[ty] = hs[after[ty] == INF ? 0 : after[ty]];
        if (in) {
#pragma unroll
            for (int ty = 0; ty < 2; ++ty) {
                const int64_t o = 6 * gt + 3 * ty + 2;
                k.nbx[o] = after[ty] == INF ? -1 : after[ty];
                k.nby[o] = after[ty] == INF ? (real)0 : ya[ty];
                if (k.right) k.right[2 * gt + ty] = after[ty] == INF ? -1 : after[ty];
            }
        }
    }
    const int n0 = carry[0], n1 = carry[1];
    const int wmx = (n0 + K - 1) / K;
    const int wmn = (n1 + K - 1) / K;
    unsigned wbase = 0;
    if (lane == 0) {
        k.n[2 * s] = n0;
        k.n[2 * s + 1] = n1;
        wbase = atomicAdd(pc.wincount, (unsigned)(wmx + wmn));
        if (dense) atomicAdd(&pc.dense[pc.epoch], dense);
    }
    wbase = (unsigned)__builtin_amdgcn_readfirstlane((int)wbase);
    wave_sync();   // the window hints written by other lanes
    for (int w = lane; w < wmx + wmn; w += kWave) {
        int type, wi;
        window_of_item(w, wmx, wmn, type, wi);
        pc.winlist[kWinItem * (wbase + w)] = s;
        pc.winlist[kWinItem * (wbase + w) + 1] = (wi << 1) | type;
        pc.winlist[kWinItem * (wbase + w) + 2] = wi < kPWin ? s_hint[wv][type][wi] : -1;
    }
}

// ------------------------------------------------------- windowed spline solve

// Positions of knots [glo, ghi) of (series s, type) into LDS (sp index =
// g - lo), from the tile bitmasks (mask [tile][type][row]), knot prefixes and
// counts.  One wavefront; tpre (64 ints) and tmask (64 x 4 words) are LDS
// scratch.  Tiles are taken 64 at a time (their prefixes and masks in LDS).
// When the knots of a chunk lie in up to 40 tiles, each lane walks the set
// bits of 32 samples at a time; otherwise of its own tile (solve launches, 16
// ragged FP32 series x 100, with the line at 16 / 40 / 64 tiles: 36.2 / 35.9 /
// 36.4 ms, 36.9 when every lane of a few-tile chunk tested its own bit of each
// row; one FP64 series of 244032 x 200: 16.32 / 16.30 / 17.4, before 16.4).
// hint = the tile holding knot glo, or -1 (64-ary search).
// (inlined: as a called function it cost the solve 8 % and the adjoint
// window solve 1 %)
// row masks of one staged tile in LDS (TW words per tile).  The adjoint
// pads them from 4 to 5 words: the 64 lanes store their tiles' rows at a
// 40-byte stride instead of 32, which spreads the stores over the banks.
// The solve keeps 4: 2 KB less LDS per workgroup.
constexpr int kTMaskW = kWR + 1;

// 32 samples' bits of a row mask that was written whole
typedef uint32_t __attribute__((may_alias)) MaskHalf;

template <int TW>
__device__ __forceinline__ void gather_positions(const SeriesDev& sd, const uint64_t* kmask,
                                                 const int* kpre, const int* kcnt, int s, int type,
                                                 long lo, int glo, int ghi, int* sp, int* tpre,
                                                 uint64_t (*tmask)[TW], int hint, int n)
{
    const int lane = threadIdx.x & 63;
    const int tb = load_scalar(sd.tile0 + s), ntl = load_scalar(sd.ntl + s);
    int a = hint >= 0 ? hint : 0, b = hint >= 0 ? hint + 1 : ntl;
    while (b - a > 1) {
        const int step = (b - a + kWave - 1) / kWave;
        const int idx = a + lane * step;
        const bool ok = idx < b && kpre[2 * (tb + idx) + type] <= glo;
        const uint64_t m = wave_ballot(ok);
        const int L = 63 - __builtin_clzll(m);
        a = a + L * step;
        b = min(a + step, b);
    }
    int g = glo;
    int tile = a;
    // the lane's tile of a chunk: prefix, count, row masks
    struct Chunk {
        int p, c;
        uint64_t mk[kWR];
    };
    auto request = [&](int first, Chunk& q) {
        const int tl = first + lane;
        const bool valid = tl < ntl;
        q.p = valid ? kpre[2 * (tb + tl) + type] : 0x7FFFFFFF;
        q.c = valid ? kcnt[2 * (tb + tl) + type] : 0;
#pragma unroll
        for (int r = 0; r < kWR; ++r) q.mk[r] = valid ? kmask[8 * (int64_t)(tb + tl) + kWR * type + r] : 0ull;
    };
    Chunk cur, nxt;
    request(tile, cur);
    const bool sparse = (int64_t)(ghi - glo) * ntl > (int64_t)n * kWave;
    while (g < ghi) {
        // where a window spans more than one chunk, the next is requested
        // before this one is waited for (FP32 solve launches 35.9 -> 35.8 ms,
        // FP64 16.30 -> 16.20)
        const int tl = tile + lane;
        const bool valid = tl < ntl;
        const bool ahead = sparse && tile + kWave < ntl;
        if (ahead) request(tile + kWave, nxt);
        const int p = cur.p, c = cur.c;
        uint64_t mk[kWR];
#pragma unroll
        for (int r = 0; r < kWR; ++r) mk[r] = cur.mk[r];
        tpre[lane] = p;
#pragma unroll
        for (int r = 0; r < kWR; ++r) tmask[lane][r] = mk[r];
        const uint64_t vm = wave_ballot(valid);
        if (vm == 0ull) break;   // counts inconsistent with n: leave the rest
        const int last = 63 - __builtin_clzll(vm);
        const int pend = __shfl(p + c, last, kWave);
        const int gend = min(ghi, pend);
        // chunk tiles holding the first and the last knot of [g, gend)
        const uint64_t ua = vm & wave_ballot(p <= g), ub = vm & wave_ballot(p <= gend - 1);
        const int xa = ua ? 63 - __builtin_clzll(ua) : 0;
        const int xb = ub ? 63 - __builtin_clzll(ub) : 0;
        wave_sync();
        if (xb - xa < 40) {
            // a lane per 32 samples: it walks the set bits of its word, from
            // the rank that its tile's prefix and the words before it give
            for (int q0 = 8 * xa; q0 <= 8 * xb; q0 += kWave) {
                const int x = (q0 + lane) >> 3, sub = lane & 7;
                const bool in = x <= xb;
                uint32_t m = in ? ((const MaskHalf*)tmask[in ? x : 0])[sub] : 0u;
                int before = __popc(m);
                int gi = (in ? tpre[in ? x : 0] : 0) - before;
                const int s1 = dpp_row_i<0x111, 0xF>(before, 0);
                before += sub >= 1 ? s1 : 0;
                const int s2 = dpp_row_i<0x112, 0xF>(before, 0);
                before += sub >= 2 ? s2 : 0;
                const int s4 = dpp_row_i<0x114, 0xF>(before, 0);
                before += sub >= 4 ? s4 : 0;
                gi += before;
                const int pos = (tile + x) * kWT + 32 * sub;
                while (m != 0u) {
                    const int bit = __builtin_ctz(m);
                    m &= m - 1u;
                    if ((unsigned)(gi - g) < (unsigned)(gend - g)) sp[gi - lo] = pos + bit;
                    ++gi;
                }
            }
        } else if (lane >= xa && lane <= xb) {
            // many tiles with few knots each: every lane walks the set bits
            // of its own tile (prefix and row masks still in its registers)
            int gi = p;
#pragma unroll
            for (int r = 0; r < kWR; ++r) {
                uint64_t m = mk[r];
                while (m != 0ull && gi < gend) {
                    const int bit = __builtin_ctzll(m);
                    m &= m - 1ull;
                    if (gi >= g) sp[gi - lo] = (tile + lane) * kWT + kWave * r + bit;
                    ++gi;
                }
            }
        }
        g = gend;
        tile += kWave;
        wave_sync();
        if (ahead) cur = nxt;
        else if (g < ghi) request(tile, cur);
    }
}

// Values of knots [glo, ghi) (positions already in sp) from the series' pass
// input hs (N samples) into sy; every load is issued before any store.
template <typename real, int NIT>
__device__ void gather_values(const real* hs, int N, long lo, int glo, int ghi, const int* sp,
                              real* sy)
{
    const int lane = threadIdx.x & 63;
    for (int i0 = (int)(glo - lo); i0 < (int)(ghi - lo); i0 += kWave * NIT) {
        int pos[NIT];
#pragma unroll
        for (int j = 0; j < NIT; ++j) {
            const int i = i0 + lane + kWave * j;
            pos[j] = i < ghi - lo ? min(max(sp[i], 0), N - 1) : -1;
        }
        real yv[NIT];
#pragma unroll
        for (int j = 0; j < NIT; ++j) yv[j] = pos[j] >= 0 ? hs[pos[j]] : (real)0;
#pragma unroll
        for (int j = 0; j < NIT; ++j) {
            const int i = i0 + lane + kWave * j;
            if (pos[j] >= 0) sy[i] = yv[j];
        }
    }
}

// One wavefront per window item.  NAK = not-a-knot ends, as its own
// instance: the natural-end instance carries no end-row divisions (FP64:
// 113 registers, four waves per SIMD; the not-a-knot one 149, three).
template <typename real, int B, int H, bool NAK>
__global__ __launch_bounds__(kThreads) void k_solve(SolveArgs<real> a)
{
    constexpr int W = kWave * B;
    constexpr int K = W - 2 * H;
    constexpr int NW = kThreads / kWave;
    // rows padded to a multiple of 16 bytes, so a lane's B + 2 entries at
    // r = lane * B start 16-byte aligned
    __shared__ __align__(16) int s_pos[NW][W + 4];
    __shared__ __align__(16) real s_y[NW][W + 4];
    __shared__ int s_tpre[NW][kWave];
    __shared__ uint64_t s_tmask[NW][kWave][kWR];
    const int wv = wave_index(), lane = threadIdx.x & 63;
    int* sp = s_pos[wv];
    real* sy = s_y[wv];
    // window items and series metadata through the scalar cache (written
    // by earlier launches): one round trip for the item, one for its series
    if (a.run && load_scalar(a.run) == 0u) return;
    const unsigned total = load_scalar(a.wincount);
    for (unsigned item = blockIdx.x * NW + wv; item < total; item += gridDim.x * NW) {
        const int s = load_scalar(a.winlist + kWinItem * item);
        const int code = load_scalar(a.winlist + kWinItem * item + 1);
        const int hint = load_scalar(a.winlist + kWinItem * item + 2);
        const int type = code & 1;
        const int w = code >> 1;
        if (a.active && !load_scalar(a.active + s)) continue;
        const int n = load_scalar(a.k.n + 2 * s + type);
        const int64_t kb = load_scalar(a.sd.kbase + s) + (type ? a.sd.kstride : 0);
        const long g0 = (long)w * K - H;
        const long lo = g0 - 1;
        const int glo = (int)max(lo, 0L);
        const int ghi = (int)min(lo + W + 2, (long)n);
        constexpr int NIT = (W + 2 + kWave - 1) / kWave;
        gather_positions<kWR>(a.sd, a.k.mask, a.k.pre, a.k.cnt, s, type, lo, glo, ghi, sp,
                              s_tpre[wv], s_tmask[wv], hint, n);
        wave_sync();
        gather_values<real, NIT>(a.h + load_scalar(a.sd.off + s), load_scalar(a.sd.len + s), lo, glo,
                                 ghi, sp, sy);
        wave_sync();
        // endpoint fix-up when n >= 6 (setBoundaryMax/Min, cudaICEEMDAN.cu:209-291);
        // idempotent, so every window that holds an end applies it
        if (lane == 0) {
            const long keep0 = (long)w * K;
            if (lo <= 0) {
                const int i0 = (int)(-lo);
                int replaced = 0;
                if (n >= 6) {
                    const real slope =
                        (sy[i0 + 2] - sy[i0 + 1]) / (real)(sp[i0 + 2] - sp[i0 + 1]);
                    const real t = sy[i0 + 1] - slope * (real)(sp[i0 + 1] - sp[i0]);
                    if (type == 0 ? (t > sy[i0]) : (t < sy[i0])) {
                        sy[i0] = t;
                        replaced = 1;
                    }
                }
                if (w == 0) {
                    a.k.fix[4 * s + 2 * type] = sy[i0];
                    if (a.fixf) a.fixf[4 * s + 2 * type] = replaced;
                }
            }
            const long ie = (long)(n - 1) - lo;
            if (ie >= 0 && ie < W + 2) {
                const int i1 = (int)ie;
                int replaced = 0;
                if (n >= 6) {
                    const real slope =
                        (sy[i1 - 1] - sy[i1 - 2]) / (real)(sp[i1 - 1] - sp[i1 - 2]);
                    const real t = sy[i1 - 1] + slope * (real)(sp[i1] - sp[i1 - 1]);
                    if (type == 0 ? (t > sy[i1]) : (t < sy[i1])) {
                        sy[i1] = t;
                        replaced = 1;
                    }
                }
                if (n - 1 >= keep0 && n - 1 < keep0 + K) {
                    a.k.fix[4 * s + 2 * type + 1] = sy[i1];
                    if (a.fixf) a.fixf[4 * s + 2 * type + 1] = replaced;
                }
            }
        }
        wave_sync();

        // the lane's rows r = rb .. rb+B-1 (LDS index r + 1) need window
        // knots rb .. rb+B+1: loaded once, as wide reads, and the B + 1
        // intervals between them give every row its lengths and slopes
        const int rb = lane * B;
        int hx[B + 1];
        real sl[B + 1];
        {
            int px[B + 2];
            real py[B + 2];
#pragma unroll
            for (int j = 0; j < B + 2; ++j) {
                px[j] = sp[rb + j];
                py[j] = sy[rb + j];
            }
#pragma unroll
            for (int j = 0; j <= B; ++j) {
                hx[j] = px[j + 1] - px[j];
                sl[j] = sdiv<real>(py[j + 1] - py[j], (real)hx[j]);
            }
        }
        real xs[B];
        partition_pcr<real, B, !NAK>(
            lane,
            [&](int q, real& dl, real& d, real& du, real& f) {
                spline_row<real, NAK>(n, g0 + rb + q, hx[q], hx[q + 1], sl[q], sl[q + 1], dl, d, du,
                                      f);
            },
            xs);
        real* cout = a.c + kb;
        const bool nak = NAK && n >= 4;
#pragma unroll
        for (int q = 0; q < B; ++q) {
            const int r = rb + q;
            const long gg = g0 + r;
            if (r >= H && r < H + K && gg < n) {
                if (!(nak && (gg == 0 || gg == n - 1))) cout[gg] = xs[q];
            }
        }
        if (nak) {
            // the window that keeps an end knot recovers it from its own rows
            wave_sync();
#pragma unroll
            for (int q = 0; q < B; ++q) sy[rb + q + 1] = xs[q];
            wave_sync();
            if (lane == 0) {
                const long r0 = -g0, r1 = (long)(n - 1) - g0;
                if (r0 >= H && r0 < H + K) {
                    const int i0 = (int)r0 + 1;
                    cout[0] = nak_end<real>(sy[i0 + 1], sy[i0 + 2], sp[i0 + 1] - sp[i0],
                                            sp[i0 + 2] - sp[i0 + 1]);
                }
                if (r1 >= H && r1 < H + K) {
                    const int i1 = (int)r1 + 1;
                    cout[n - 1] = nak_end<real>(sy[i1 - 1], sy[i1 - 2], sp[i1] - sp[i1 - 1],
                                                sp[i1 - 1] - sp[i1 - 2]);
                }
            }
        }
        wave_sync();
    }
}

// ------------------------------------------------------------ Rilling decide

// siftingCriterion (cudaICEEMDAN.cu:494-525) + checkBreak (:546-580) with
// per-series masks: export at the first stop or at pass cap-1.
template <typename real>
__global__ void k_rilling_decide(SeriesDev sd, const int* nk, const int* sx_cnt,
                                 const int* sx_mark, int* active, int* stop_pass, int* subs,
                                 int pass, int cap, const unsigned* run, unsigned* n_active)
{
    const int s = blockIdx.x;
    const int lane = threadIdx.x;
    if (load_scalar(run) == 0u) return;
    if (!active[s]) return;
    long long c = 0;
    int mk = 0;
    const int t0 = sd.tile0[s], nt = sd.ntl[s];
    for (int t = lane; t < nt; t += kWave) {
        c += sx_cnt[t0 + t];
        mk |= sx_mark[t0 + t];
    }
    for (int o = 32; o >= 1; o >>= 1) {
        c += __shfl_xor(c, o, kWave);
        mk |= __shfl_xor(mk, o, kWave);
    }
    if (lane == 0) {
        const int N = sd.len[s];
        const real frac = (real)c * (real)(1.0 / (double)N);
        const bool cont = (frac > (real)0.05) || (mk && (nk[2 * s] + nk[2 * s + 1]) > 6);
        if (!cont || pass == cap - 1) {
            active[s] = 0;
            stop_pass[s] = pass;
        } else {
            subs[s] += 1;
            atomicAdd(n_active, 1u);
        }
    }
}

// --------------------------------------------------------------- statistics

// Canonical sum: lane l of 1024 adds x[l], x[l+1024], ... in order, then a
// pairwise tree (same order as the oracle).  One workgroup per series.
// The tree: the first wave's lane t combines the 16 partial sums of stride
// 64 itself (strides 512 .. 64), then six steps inside the wave: two
// workgroup barriers instead of one per level.
template <typename real>
__device__ __forceinline__ real canon_sum_block(real acc, real* sred)
{
    const int tid = threadIdx.x;
    sred[tid] = acc;
    __syncthreads();
    if (tid < kWave) {
        real v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = sred[tid + kWave * q];
#pragma unroll
        for (int st = 8; st >= 1; st >>= 1)
#pragma unroll
            for (int q = 0; q < st; ++q) v[q] = v[q] + v[q + st];
        real r = v[0];
#pragma unroll
        for (int st = 32; st >= 1; st >>= 1) r = r + shfl_down(r, st);
        if (tid == 0) sred[0] = r;
    }
    __syncthreads();
    const real r = sred[0];
    __syncthreads();
    return r;
}

// Sum over p = tid, tid + 1024, ... < N of f(loaded values), in order, the
// loads of kSumAhead terms requested before the first is added: a lane's
// chain is N / 1024 dependent adds, which took one memory round trip each
// (244032 FP32 samples: 114 us for both passes of the variance).
constexpr int kSumAhead = 16;
template <typename real, class Load, class Term>
__device__ __forceinline__ real canon_lane_sum(int N, Load load, Term term)
{
    real acc = (real)0;
    int p = threadIdx.x;
    for (; p + 1024 * (kSumAhead - 1) < N; p += 1024 * kSumAhead) {
        decltype(load(0)) v[kSumAhead];
#pragma unroll
        for (int q = 0; q < kSumAhead; ++q) v[q] = load(p + 1024 * q);
#pragma unroll
        for (int q = 0; q < kSumAhead; ++q) acc = acc + term(v[q]);
    }
    // the last terms at clamped indices, so that their loads go out together
    if (p < N) {
        decltype(load(0)) v[kSumAhead];
#pragma unroll
        for (int q = 0; q < kSumAhead; ++q) v[q] = load(min(p + 1024 * q, N - 1));
#pragma unroll
        for (int q = 0; q < kSumAhead; ++q)
            if (p + 1024 * q < N) acc = acc + term(v[q]);
    }
    return acc;
}

// Mean and unbiased variance (two passes) of every series, one workgroup
// each; optionally the scale a stage start multiplies the noise with, as
// double: 1 / std (SCALE_INV) or std (SCALE_STD).
template <typename real>
__global__ __launch_bounds__(1024) void k_series_var(const real* base, const int64_t* off,
                                                     int64_t stride, const int* len, real* var_out,
                                                     real* mean_out, double* scale_out, int scale)
{
    __shared__ real sred[1024];
    const int s = blockIdx.x;
    const int64_t o = off ? off[s] : (int64_t)s * stride;
    const real* x = base + o;
    const int N = len ? len[s] : (int)stride;
    auto at = [&](int p) { return x[p]; };
    const real mu = canon_sum_block<real>(canon_lane_sum<real>(N, at, [](real v) { return v; }), sred) *
                    (real)(1.0 / (double)N);
    const real ss = canon_sum_block<real>(canon_lane_sum<real>(N, at, [&](real v) {
                                              const real dv = v - mu;
                                              return dv * dv;
                                          }), sred);
    if (threadIdx.x == 0) {
        const real var = ss * (real)(1.0 / (double)(N - 1));
        if (var_out) var_out[s] = var;
        if (mean_out) mean_out[s] = mu;
        if (scale_out) {
            const real sd = sqrt(var);
            scale_out[s] = scale == SCALE_STD ? (double)sd : 1.0 / (double)sd;
        }
    }
}

// ------------------------------------------------- sift pass, wave per tile
// One wavefront sifts a run of consecutive 256-sample tiles of one series;
// lane l owns samples t0 + 64 r + l, r = 0..3.  Everything a tile needs is
// wave-local: the knot flags of h are ballots (their ranks give each
// sample's interval), the knot table [pre-2, pre+cnt] of both types lives in
// the wave's own LDS slice, and no workgroup barrier is used, so the four
// waves of a workgroup run independent segments.

// Lane 0 stores the eight wave-uniform row masks m[type][row] (no lane-
// dependent indexing, which would put the array in scratch memory).
__device__ __forceinline__ void store_masks(uint64_t* dst, const uint64_t (&m)[2][kWR], int lane)
{
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < 2 * kWR; ++q) dst[q] = m[q / kWR][q % kWR];
    }
}

// Per-wave knot table of a tile (KC entries per type): each knot's position
// and the coefficients of the interval that starts at it.  The small
// tables keep one record per knot (coefficients, then the position: 32
// bytes in FP32, 48 in FP64), so that a knot's position and coefficients
// are read at one LDS address (-2.5 % on the FP32 sift, -1 % on FP64); the
// full tables keep two arrays (records would cost them waves per SIMD:
// their LDS would grow from 22 to 35 KB per workgroup in FP32, to 52 KB in
// FP64).
// Positions are relative to the tile.  The small FP64 table keeps them as
// doubles, so that t = p - pos is one subtraction; the full one keeps integers
// (doubles would cost it a wave per SIMD), and so does FP32, where a float
// holds no position 2^24 samples away (floats were 1 % faster).
template <typename real, int KC, bool REC>
struct KnotTableOf {
    using pos_t = int;
    pos_t pos[2][KC];
    Coef<real> q[2][KC];
    __device__ __forceinline__ pos_t& P(int ty, int j) { return pos[ty][j]; }
    __device__ __forceinline__ Coef<real>& Q(int ty, int j) { return q[ty][j]; }
};
template <typename real, int KC>
struct KnotTableOf<real, KC, true> {
    using pos_t = typename std::conditional<std::is_same<real, double>::value, double, int>::type;
    struct alignas(sizeof(real) == 4 ? 32 : 16) Rec {
        Coef<real> q;
        pos_t pos;
    };
    Rec r[2][KC];
    __device__ __forceinline__ pos_t& P(int ty, int j) { return r[ty][j].pos; }
    __device__ __forceinline__ Coef<real>& Q(int ty, int j) { return r[ty][j].q; }
};
template <typename real, int KC>
using KnotTable = KnotTableOf<real, KC, KC == kWKS>;

// Which samples of a tile a lane of the sift holds: the four from 4 lane in
// FP32 (one 16-byte load and store, neighbours mostly in the lane itself,
// ranks and mask bits shared by its four samples), sample 64 q + lane of each
// row q in FP64, where quads would be 32 bytes apart in every access.  Sift
// launches of both dtypes in milliseconds (16 ragged FP32 series of 8192 ..
// 262144 samples x 100; one FP64 series of 244032 x 200): rows 112.8 and
// 42.4, quads 107.5 and 47.3 to 52.
template <typename real>
struct Lay {
    static constexpr bool kQuad = sizeof(real) == 4;
    __device__ __forceinline__ static int at(int q, int lane) { return kQuad ? 4 * lane + q : kWave * q + lane; }
};

// NT: samples go past the caches in both directions, as a pass reads and writes
// each once; what is read again (tables, masks) stays cached (sift launches
// above with rows: 114.3 -> 112.8 ms FP32, 44.5 -> 42.5 FP64).  Only where the
// samples do not fit the caches (sift_past_caches): the passes and knot
// prefixes of a smaller phase read them there (96 MB of FP64 samples, Rilling
// rule, 91.1 ms past the caches, 85.2 through them).  A whole tile's samples of
// the lane, a series may start at any sample.
typedef float Quad __attribute__((ext_vector_type(4), aligned(4)));
template <bool NT, typename T>
__device__ __forceinline__ T load_sample(const T* p)
{
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}
template <bool NT, typename T>
__device__ __forceinline__ void store_sample(T v, T* p)
{
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}
template <bool NT, typename real>
__device__ __forceinline__ void load_quad(const real* p, real (&v)[kWR])
{
    const Quad q = load_sample<NT>((const Quad*)p);
#pragma unroll
    for (int i = 0; i < kWR; ++i) v[i] = q[i];
}
template <bool NT, typename real>
__device__ __forceinline__ void store_tile(real* p, int lane, const real (&v)[kWR])
{
    if constexpr (Lay<real>::kQuad) {
        const Quad q = {v[0], v[1], v[2], v[3]};
        store_sample<NT>(q, (Quad*)(p + 4 * lane));
    } else {
#pragma unroll
        for (int r = 0; r < kWR; ++r) store_sample<NT>(v[r], p + r * kWave + lane);
    }
}

// Knots of one type among a lane's four samples of a quad: the mask byte of
// the lane pair, and from it bit l of bm[q] for sample 4 l + q of the tile.
__device__ __forceinline__ unsigned quad_byte(const uint64_t* mask, int64_t gt, int ty, int lane)
{
    return ((const uint8_t*)(mask + 8 * gt + kWR * ty))[lane >> 1];
}
__device__ __forceinline__ void quad_masks(unsigned byte, int lane, uint64_t (&bm)[kWR])
{
    const unsigned n = byte >> ((lane & 1) * 4);
#pragma unroll
    for (int q = 0; q < kWR; ++q) bm[q] = wave_ballot((n & (1u << q)) != 0u);
}

// 2 v + bit of the lane in m, v + bit of the lane in m
__device__ __forceinline__ unsigned shift_in(unsigned v, uint64_t m)
{
    return v + v + (__builtin_amdgcn_inverse_ballot_w64(m) ? 1u : 0u);
}
__device__ __forceinline__ int add_bit(int v, uint64_t m)
{
    return v + (__builtin_amdgcn_inverse_ballot_w64(m) ? 1 : 0);
}

// lanes whose sample q of a tile with nt samples is inside the series, and
// those where it is one of the series' two ends (left = samples from the
// tile's start to the series' end)
template <typename real>
__device__ __forceinline__ void lay_ends(int q, int nt, bool first, int left, uint64_t& valid, uint64_t& end)
{
    const int in = Lay<real>::kQuad ? (nt - q + kWR - 1) / kWR : min(max(nt - q * kWave, 0), kWave);
    valid = in >= kWave ? ~0ull : (1ull << in) - 1;
    end = first && q == 0 ? 1ull : 0ull;
    const int last = left - 1;
    const int lq = Lay<real>::kQuad ? last % kWR : last / kWave, ll = Lay<real>::kQuad ? last / kWR : last % kWave;
    if (left <= kWT && lq == q) end |= 1ull << ll;
}

template <typename real, int KC>
struct WTile {
    static constexpr int NC = (KC + kWave - 1) / kWave;
    real h[kWR];
    real c[2][NC];        // c of knots pre-2+j, j = lane + 64 k
    int nbx;
    real nby;             // lanes 0..5: values of knots pre-1, pre-2, pre+cnt per type
    // knots of h: of the lane's quad, bits 4 (lane & 1) .. of the type's byte;
    // else lanes 0..7: row masks [type][row] (other lanes: copies)
    typename std::conditional<Lay<real>::kQuad, unsigned[2], uint64_t>::type mk;
};

// One segment of tiles, sifted by one wavefront with a knot table of KC
// entries per type.  A tile whose knots do not fit (cnt + 3 > KC) is an error
// with the full table (KC = kWKC fits every tile); with the small table it is
// appended to a.ovf_segs for a second launch with the full table, and the
// tile after it takes h_new of its left neighbour from its own knots.
//
// The pass is bound by the number of instructions of all kinds: VALU, scalar
// and memory pipes were each about 58 % busy, and more than six waves per SIMD
// changed nothing.
template <typename real, bool RILL, int KC, bool NT>
__device__ __forceinline__ void sift_segment(const SiftArgs<real>& a, const Segment* segs, int sid,
                                             int lane, KnotTable<real, KC>& T)
{
    const SeriesDev& sd = a.sd;
    const Segment seg = segs[sid];
    const int s = seg.s;
    if (a.active && !a.active[s]) return;
    const int N = sd.len[s];
    const int tb = sd.tile0[s];
    const real* h = a.h_in + sd.off[s];
    real* hout = a.h_out + sd.off[s];
    const int nn[2] = {a.kin.n[2 * s], a.kin.n[2 * s + 1]};
    const real* cp[2] = {a.c + sd.kbase[s], a.c + sd.kstride + sd.kbase[s]};
    // end-knot values after the endpoint fix, first and last, of the type of
    // this lane's neighbour knot (lanes 0..2 maxima, 3..5 minima)
    const real fx0 = a.kin.fix[4 * s + (lane >= 3 ? 2 : 0)], fx1 = a.kin.fix[4 * s + (lane >= 3 ? 3 : 1)];
    const bool use_mean = (nn[0] > 3) && (nn[1] > 3);
    using pos_t = typename KnotTable<real, KC>::pos_t;

    int mpre[2], mcnt[2];
    auto meta_ints = [&](int64_t gt, int (&pre)[2], int (&cnt)[2]) {
        pre[0] = load_scalar(a.kin.pre + 2 * gt);
        pre[1] = load_scalar(a.kin.pre + 2 * gt + 1);
        cnt[0] = load_scalar(a.kin.cnt + 2 * gt);
        cnt[1] = load_scalar(a.kin.cnt + 2 * gt + 1);
    };

    auto load = [&](int t, const int (&pre)[2], const int (&cnt)[2], WTile<real, KC>& w) {
        const int t0 = t * kWT;
        if (Lay<real>::kQuad && t0 + kWT <= N) {
            load_quad<NT>(h + t0 + 4 * lane, w.h);
        } else {
#pragma unroll
            for (int q = 0; q < kWR; ++q) {
                const int p = t0 + Lay<real>::at(q, lane);
                w.h[q] = p < N ? load_sample<NT>(h + p) : (real)0;
            }
        }
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            // (entries outside the series are never used)
#pragma unroll
            for (int k = 0; k < WTile<real, KC>::NC; ++k) {
                const int j = lane + k * kWave;
                w.c[ty][k] = (real)0;
                if (j < cnt[ty] + 3) w.c[ty][k] = cp[ty][min(max(pre[ty] - 2 + j, 0), nn[ty] - 1)];
            }
        }
        w.nbx = -1;
        w.nby = (real)0;
        if (lane < 6) {
            const int64_t o = 6 * (int64_t)(tb + t) + lane;
            w.nbx = a.kin.nbx[o];
            w.nby = a.kin.nby[o];
        }
        if constexpr (Lay<real>::kQuad) {
            w.mk[0] = quad_byte(a.kin.mask, tb + t, 0, lane);
            w.mk[1] = quad_byte(a.kin.mask, tb + t, 1, lane);
        } else {
            w.mk = a.kin.mask[8 * (int64_t)(tb + t) + (lane & 7)];
        }
    };

    int npre[2] = {0, 0}, ncnt[2] = {0, 0};
    meta_ints(tb + seg.t_first, mpre, mcnt);
    WTile<real, KC> cur, nxt;
    load(seg.t_first, mpre, mcnt, cur);
    // the sample just before the tile: h' of it where `carry` (the previous
    // tile of the segment computed it: same interval, same coefficients, same
    // bits), else h
    real edge = seg.t_first > 0 ? h[seg.t_first * kWT - 1] : (real)0;
    bool carry = false;
    // the first tile is needed at once; waiting here also tells the compiler
    // that nothing loaded before the loop is outstanding inside it, so the
    // loop body never waits on the prefetch of the next tile
    wait_vmem();
    // The last sample of a tile has its right neighbour in the next one: it is
    // stored as no knot and added when that tile's h' is known (by lane 0),
    // instead of evaluating the neighbour with this tile's table as well.
    // open: bit 0 = such a sample waits, bit 1 (2) = the sample before it is
    // greater (less).
    unsigned open = 0;
    auto close = [&](int gt, unsigned o, unsigned g, unsigned l) {
        const unsigned bx = (o >> 2) & g, bn = (o >> 1) & l;
        if (((bx | bn) & 1u) && lane == 0) {
            const int64_t w = 2 * (int64_t)gt + (bn & 1u);
            atomicOr((unsigned*)(a.kout.mask + kWR * w + kWR - 1) + 1, 0x80000000u);
            atomicAdd(a.kout.cnt + w, 1);
        }
    };

    for (int i = 0; i < seg.count; ++i) {
        const int t = seg.t_first + i;
        const int gt = tb + t;
        const int t0 = t * kWT;
        const int nt = min(kWT, N - t0);
        const int pre[2] = {mpre[0], mpre[1]}, cnt[2] = {mcnt[0], mcnt[1]};
        // the next tile does not follow here: this one closes its own end
        bool tail = true;
        if (i + 1 < seg.count) {
            meta_ints(gt + 1, npre, ncnt);
            tail = ncnt[0] + 3 > KC || ncnt[1] + 3 > KC;
            load(t + 1, npre, ncnt, nxt);
        }

        // ---- knot flags of h (find_extrema_shfl_*, cudaICEEMDAN.cu:92-148):
        // the previous pass (or the stage start) found them when it wrote h,
        // from the same neighbour values, and stored them as bitmasks; bm[ty][q]
        // has bit l for sample q of lane l
        uint64_t bm[2][kWR];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            if constexpr (Lay<real>::kQuad) {
                quad_masks(cur.mk[ty], lane, bm[ty]);
            } else {
#pragma unroll
                for (int q = 0; q < kWR; ++q) bm[ty][q] = lane_value(cur.mk, ty * kWR + q);
            }
        }
        const bool over = cnt[0] + 3 > KC || cnt[1] + 3 > KC;
        int tot[2];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty)
            tot[ty] = __popcll(bm[ty][0]) + __popcll(bm[ty][1]) + __popcll(bm[ty][2]) + __popcll(bm[ty][3]);
        if (tot[0] != cnt[0] || tot[1] != cnt[1] || (over && !a.ovf_segs)) {
            if (lane == 0) atomicOr(a.pc.err, ICM_DEVERR_KNOTCAP);
            return;
        }

        // interior tiles (neither series end inside, all 256 samples valid)
        // take a copy of the body without the per-lane end tests
        auto tile = [&](auto full_c) {
            constexpr bool FULL = decltype(full_c)::value;
            // interval (table index) of every sample of the lane: knots
            // strictly before it, less one; a knot's own entry is the next
            int iv[2][4];
#pragma unroll
            for (int ty = 0; ty < 2; ++ty) {
                int v = 1;
                if constexpr (Lay<real>::kQuad) {
#pragma unroll
                    for (int q = 0; q < kWR; ++q) v = rank_below(bm[ty][q], v);
                    iv[ty][0] = v;
#pragma unroll
                    for (int q = 0; q < kWR - 1; ++q) iv[ty][q + 1] = add_bit(iv[ty][q], bm[ty][q]);
                } else {
#pragma unroll
                    for (int q = 0; q < kWR; ++q) {
                        iv[ty][q] = rank_below(bm[ty][q], v);
                        v += __popcll(bm[ty][q]);
                    }
                }
            }
            // ---- knot table: index j <-> knot pre - 2 + j
            if (FULL && Lay<real>::kQuad) {
                // of two neighbouring samples at most one is a maximum (minimum)
#pragma unroll
                for (int q = 0; q < 4; q += 2) {
#pragma unroll
                    for (int ty = 0; ty < 2; ++ty) {
                        if (__builtin_amdgcn_inverse_ballot_w64(bm[ty][q] | bm[ty][q + 1])) {
                            const bool second = __builtin_amdgcn_inverse_ballot_w64(bm[ty][q + 1]);
                            const int j = iv[ty][q] + 1;
                            T.P(ty, j) = (pos_t)(4 * lane + q + (second ? 1 : 0));
                            T.Q(ty, j).a = second ? cur.h[q + 1] : cur.h[q];
                        }
                    }
                }
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int ty = 0; ty < 2; ++ty) {
                        if (__builtin_amdgcn_inverse_ballot_w64(bm[ty][q])) {
                            const int j = iv[ty][q] + 1;
                            const int g = pre[ty] - 2 + j;
                            real y = cur.h[q];
                            if (!FULL) {   // knots 0 and n-1 lie in the series' end tiles
                                if (g == 0) y = lane_value(fx0, 3 * ty);
                                if (g == nn[ty] - 1) y = lane_value(fx1, 3 * ty);
                            }
                            T.P(ty, j) = (pos_t)Lay<real>::at(q, lane);
                            T.Q(ty, j).a = y;
                        }
                    }
                }
            }
            if (lane < 6) {
                const int ty = lane / 3, w = lane % 3;
                const int j = w == 0 ? 1 : (w == 1 ? 0 : cnt[ty] + 2);
                const int g = pre[ty] - 2 + j;
                if (cur.nbx >= 0 && g >= 0 && g < nn[ty]) {
                    real y = cur.nby;
                    if (g == 0) y = fx0;
                    if (g == nn[ty] - 1) y = fx1;
                    T.P(ty, j) = (pos_t)(cur.nbx - t0);
                    T.Q(ty, j).a = y;
                }
            }
#pragma unroll
            for (int ty = 0; ty < 2; ++ty)
#pragma unroll
                for (int k = 0; k < WTile<real, KC>::NC; ++k) {
                    const int j = lane + k * kWave;
                    if (j < cnt[ty] + 3) T.Q(ty, j).c = cur.c[ty][k];
                }
            wave_sync();
            // ---- interval coefficients (spline_coefficients, cudaICEEMDAN.cu:394-398)
            // both types in one strided loop (intervals j of type 0, then of type 1)
            for (int q = lane; q < cnt[0] + cnt[1] + 4; q += kWave) {
                const int ty = q >= cnt[0] + 2;
                const int j = ty ? q - (cnt[0] + 2) : q;
                const int g = pre[ty] - 2 + j;
                if (g < 0 || g + 1 > nn[ty] - 1) continue;
                const real hk = (real)(T.P(ty, j + 1) - T.P(ty, j));
                const real a0 = T.Q(ty, j).a, a1 = T.Q(ty, j + 1).a;
                const real c0 = T.Q(ty, j).c, c1 = T.Q(ty, j + 1).c;
                interval_bd<real>(hk, a0, a1, c0, c1, T.Q(ty, j).b, T.Q(ty, j).d);
            }
            wave_sync();

            // ---- envelopes, mean, h_new = h - m (interpolate :403-439,
            // averageUppperLower :441-454, updateRealizations :527-544)
            // envelope of type ty at tile offset u, interval j of the table
            auto env = [&](int ty, int j, int u) {
                return horner(T.Q(ty, j), (real)((pos_t)u - T.P(ty, j)));
            };
            real hn[kWR] = {cur.h[0], cur.h[1], cur.h[2], cur.h[3]};
            int sxc = 0;
            bool sxm = false;
            if (RILL || use_mean) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int u = Lay<real>::at(q, lane);
                    // sample 0 of the series lies in interval 0
                    const bool p0 = !FULL && q == 0 && t0 + u == 0;
                    const real U = env(0, p0 ? 2 : iv[0][q], u), L = env(1, p0 ? 2 : iv[1][q], u);
                    if (!RILL || use_mean) hn[q] = cur.h[q] - (U + L) / (real)2;
                    if (RILL && (FULL || u < nt)) {
                        const real sx = fabs((U + L) / (U - L));
                        sxc += (sx > (real)0.05) ? 1 : 0;
                        sxm |= sx > (real)0.5;
                    }
                }
            }
            if (RILL) {
                for (int o = 32; o >= 1; o >>= 1) sxc += __shfl_xor(sxc, o, kWave);
                const uint64_t mk = wave_ballot(sxm);
                if (lane == 0) {
                    a.sx_cnt[gt] = sxc;
                    a.sx_mark[gt] = mk != 0ull ? 1 : 0;
                }
            }
            // Every store of the tile comes after this wait, which the next
            // tile's loads (requested at the start of this one) and the
            // previous tile's stores have passed by now; without it the loop
            // waits for its own stores at the latch.
            auto stores = [&]() {
                wait_vmem();
                if (FULL) {
                    store_tile<NT>(hout + t0, lane, hn);
                } else {
#pragma unroll
                    for (int q = 0; q < kWR; ++q) {
                        const int u = Lay<real>::at(q, lane);
                        if (u < nt) hout[t0 + u] = hn[q];
                    }
                }
            };

            if (a.emit) {
                // h_new of the samples beside the tile where no tile of this
                // segment has it, by every lane (same LDS words)
                real hnl = edge, hnr = (real)0;
                if (!carry && (FULL || t0 >= 1)) {
                    // a knot lies on the interval to its left
                    const int ju = T.P(0, 1) == (pos_t)-1 ? 0 : 1;
                    const int jl = T.P(1, 1) == (pos_t)-1 ? 0 : 1;
                    const real U = env(0, ju, -1), L = env(1, jl, -1);
                    hnl = edge - (use_mean ? (U + L) / (real)2 : (real)0);
                }
                if (tail && (FULL || t0 + kWT < N)) {
                    const real hr = h[t0 + kWT];
                    const real U = env(0, cnt[0] + 1, kWT), L = env(1, cnt[1] + 1, kWT);
                    hnr = hr - (use_mean ? (U + L) / (real)2 : (real)0);
                }
                // ---- knots of h_new (select_extrema_*, :150-207): their row
                // bitmasks and counts (the next pass's knots).  A comparison
                // of neighbours serves both samples; that of the tile's last
                // one is known to its tail only.
                const uint64_t known = tail ? ~0ull : ~0ull >> 1;
                uint64_t cg = wave_ballot(hnl > hn[0]) & 1ull, cl = wave_ballot(hnl < hn[0]) & 1ull;
                const unsigned eg = (unsigned)cg, el = (unsigned)cl;
                const unsigned was = open;
                unsigned before;   // the last sample but one against the last
                uint64_t em[2][kWR];
                int run[2] = {0, 0};
                if constexpr (Lay<real>::kQuad) {
                    uint64_t g[kWR], l[kWR];
                    const real nx = shift_next(hn[0], hnr);
#pragma unroll
                    for (int q = 0; q < kWR; ++q) {
                        const real rgt = q < kWR - 1 ? hn[q < kWR - 1 ? q + 1 : q] : nx;
                        g[q] = wave_ballot(hn[q] > rgt);
                        l[q] = wave_ballot(hn[q] < rgt);
                    }
                    g[kWR - 1] &= known;
                    l[kWR - 1] &= known;
                    before = (((unsigned)(g[kWR - 2] >> 63) & 1u) << 1) | (((unsigned)(l[kWR - 2] >> 63) & 1u) << 2);
                    em[0][0] = g[0] & ((l[kWR - 1] << 1) | cl);
                    em[1][0] = l[0] & ((g[kWR - 1] << 1) | cg);
#pragma unroll
                    for (int q = 1; q < kWR; ++q) {
                        em[0][q] = g[q] & l[q - 1];
                        em[1][q] = l[q] & g[q - 1];
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < kWR; ++q) {
                        const real rgt = q == kWR - 1 ? shift_next(hn[q], hnr)
                                                      : row_next(hn[q], hn[q < kWR - 1 ? q + 1 : q]);
                        uint64_t g = wave_ballot(hn[q] > rgt), l = wave_ballot(hn[q] < rgt);
                        if (q == kWR - 1) {
                            g &= known;
                            l &= known;
                            before = (((unsigned)(g >> 62) & 1u) << 1) | (((unsigned)(l >> 62) & 1u) << 2);
                        }
                        row_extrema(g, l, cg, cl, em[0][q], em[1][q]);
                    }
                }
                open = tail ? 0u : 1u | before;
#pragma unroll
                for (int q = 0; q < kWR; ++q) {
                    if (!FULL) {
                        uint64_t valid, end;
                        lay_ends<real>(q, nt, t0 == 0, N - t0, valid, end);
#pragma unroll
                        for (int ty = 0; ty < 2; ++ty) em[ty][q] = valid & (end | em[ty][q]);
                    }
#pragma unroll
                    for (int ty = 0; ty < 2; ++ty) run[ty] += __popcll(em[ty][q]);
                }
                unsigned nb[2] = {0, 0};
                if constexpr (Lay<real>::kQuad) {
                    // the lane's four bits per type, two lanes to a byte
#pragma unroll
                    for (int ty = 0; ty < 2; ++ty) {
#pragma unroll
                        for (int q = kWR - 1; q >= 0; --q) nb[ty] = shift_in(nb[ty], em[ty][q]);
                        nb[ty] |= (unsigned)dpp_next_i((int)nb[ty], 0) << 4;
                    }
                }
                stores();
                if (was) close(gt - 1, was, eg, el);
                uint64_t* mw = a.kout.mask + 8 * (int64_t)gt;
                if constexpr (Lay<real>::kQuad) {
                    if (!(lane & 1)) {
                        uint8_t* mb = (uint8_t*)mw + (lane >> 1);
                        mb[0] = (uint8_t)nb[0];
                        mb[32] = (uint8_t)nb[1];
                    }
                } else {
                    store_masks(mw, em, lane);
                }
                if (lane == 0) {
                    a.kout.cnt[2 * gt] = run[0];
                    a.kout.cnt[2 * gt + 1] = run[1];
                }
            } else {
                stores();
            }
            edge = lane_value(hn[kWR - 1], kWave - 1);
            carry = true;
        };
        if (over) {
            // left to the launch with the full table
            if (lane == 0) {
                const unsigned q = atomicAdd(a.ovf_count, 1u);
                Segment o;
                o.s = s;
                o.t_first = t;
                o.count = 1;
                o.pad = 0;
                a.ovf_segs[q] = o;
            }
            edge = lane_value(cur.h[kWR - 1], kWave - 1);
            carry = false;
        } else if (t0 > 0 && t0 + kWT < N) {
            tile(std::true_type{});
        } else {
            tile(std::false_type{});
        }
        // the table is rewritten by the next tile
        wave_sync();
        cur = nxt;
        mpre[0] = npre[0];
        mpre[1] = npre[1];
        mcnt[0] = ncnt[0];
        mcnt[1] = ncnt[1];
    }
}

// One wavefront per segment (QUEUE = false), or (QUEUE = true) a resident
// grid of wavefronts working through the pass's segments: each wave takes
// the next segment from the pass's queue (one atomic increment, requested
// while the previous segment is sifted, so its latency overlaps that
// segment's loads) until the queue is exhausted.  The queue instance keeps
// the work of a launch independent of its grid (any number of segments);
// its loop keeps ~15 more registers live than the one-segment body, so it is
// used only where the one-wave-per-segment grid would exceed a launch's
// 2^32 work-items (or when ICM_SIFT_QUEUE=1).  Workgroups of the
// one-segment grid are dispatched as slots free up, which balances uneven
// segments as well.  Registers are held to the waves per SIMD that were
// fastest, small table and full one (sift launches as above, ms: FP32 with 6
// and 4 waves 108.4, 6 and 5 106.3, 7 and 6, which spills, 113.6; FP64 with 4
// and 4 43.9, 5 and 4 42.5).
template <typename real, int KC>
constexpr int kSiftWaves = sizeof(real) == 4 ? (KC == kWKS ? 6 : 5) : (KC == kWKS ? 5 : 1);
template <typename real, bool RILL, int KC, bool NT, bool QUEUE>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kSiftWaves<real, KC>)))
void k_sift_w(SiftArgs<real> a, int nsegs)
{
    constexpr int NW = kThreads / kWave;
    __shared__ KnotTable<real, KC> s_tab[NW];
    const int lane = threadIdx.x & 63, wv = wave_index();
    if (a.pc.run && load_scalar(a.pc.run) == 0u) return;
    // a small-table pass whose input has too many over-full tiles is left
    // to k_sift_list
    if (KC == kWKS && load_scalar(a.dense) > a.dense_max) return;
    if (!QUEUE) {
        const int sid = blockIdx.x * NW + wv;
        if (sid < nsegs)
            sift_segment<real, RILL, KC, NT>(a, a.segs, sid, lane, s_tab[wv]);
        return;
    }
    unsigned got = lane == 0 ? atomicAdd(a.queue, 1u) : 0u;
    int sid = __builtin_amdgcn_readlane((int)got, 0);
    while (sid < nsegs) {
        const unsigned next = lane == 0 ? atomicAdd(a.queue, 1u) : 0u;
        sift_segment<real, RILL, KC, NT>(a, a.segs, sid, lane, s_tab[wv]);
        wave_sync();
        sid = __builtin_amdgcn_readlane((int)next, 0);
    }
}

// Second launch of a small-table pass, with full tables, as a grid-stride
// loop: the tiles the small-table launch listed (*a.ovf_count one-tile
// segments in a.ovf_segs) or, when the pass input had too many over-full
// tiles for it to run, every segment of the pass.
template <typename real, bool RILL, bool NT>
__global__ __launch_bounds__(kThreads) void k_sift_list(SiftArgs<real> a, int nsegs)
{
    constexpr int NW = kThreads / kWave;
    __shared__ KnotTable<real, kWKC> s_tab[NW];
    const int lane = threadIdx.x & 63, wv = wave_index();
    if (a.pc.run && load_scalar(a.pc.run) == 0u) return;
    const bool all = load_scalar(a.dense) > a.dense_max;
    const Segment* segs = all ? a.segs : a.ovf_segs;
    const int ns = all ? nsegs : (int)load_scalar(a.ovf_count);
    SiftArgs<real> b = a;
    b.ovf_segs = nullptr;   // full tables hold every tile
    for (int sid = blockIdx.x * NW + wv; sid < ns; sid += gridDim.x * NW)
        sift_segment<real, RILL, kWKC, NT>(b, segs, sid, lane, s_tab[wv]);
}

// Stage start for 256-sample tiles: forms x_i and stores its knots as bitmasks.  MODE is ia.mode as a
// compile-time constant: one straight-line body per mode.
//
// Per-series pointers and scales of the tile being formed.
template <typename real, int MODE>
struct InitSeries {
    using P = typename Promote<real>::type;
    int tile0, tend, N;     // first tile, one past the last, samples
    const real* src;        // INIT_COPY / INIT_KNOTS / INIT_RESID
    const real* base;       // INIT_STAGE0 / INIT_STAGEK: the channel's signal
    const real* E;
    P scl0;
    real sclk;
    real* out;
    real* resid;
};

template <typename real, int MODE>
__device__ __forceinline__ InitSeries<real, MODE> init_series(const SeriesDev& sd,
                                                             const InitArgs<real>& ia,
                                                             real* h_out, int s)
{
    using P = typename Promote<real>::type;
    InitSeries<real, MODE> q{};
    q.tile0 = sd.tile0[s];
    q.tend = q.tile0 + sd.ntl[s];
    q.N = sd.len[s];
    const int64_t off = sd.off[s];
    q.out = (MODE == INIT_KNOTS || !h_out) ? nullptr : h_out + off;
    q.resid = MODE == INIT_RESID ? ia.resid + off : nullptr;
    if (MODE == INIT_COPY || MODE == INIT_KNOTS) {
        q.src = ia.src + off;
    } else if (MODE == INIT_RESID) {
        q.src = ia.src + off;
        q.E = ia.E + off;
    } else {
        const int c = sd.chan[s];
        q.base = ia.chan_sig + ia.chan_off[c];
        q.E = ia.E + sd.eoff[s];
        if (MODE == INIT_STAGE0) q.scl0 = (P)ia.scale[sd.nidx[s]];
        else q.sclk = (real)ia.scale[c];
    }
    return q;
}

// x_i of one tile (lane l: samples t0 + 64 r + l) and the samples just
// outside it; loads at clamped indices, then selects (a load under a lane
// condition would sit in its own block, waited for at its end)
template <typename real>
struct InitTile {
    real x[kWR];
    real xl, xr;
};

template <typename real, int MODE>
__device__ __forceinline__ void init_load(const InitSeries<real, MODE>& q, const InitArgs<real>& ia,
                                          int gt, int lane, InitTile<real>& w)
{
    using P = typename Promote<real>::type;
    const int t0 = (gt - q.tile0) * kWT;
    const int nt = min(kWT, q.N - t0);
    auto val = [&](int p) -> real {
        if (MODE == INIT_COPY || MODE == INIT_KNOTS) return q.src[p];
        if (MODE == INIT_RESID) return q.src[p] - q.E[p];
        const real e = q.E[p];
        if (MODE == INIT_STAGE0) return (real)((P)q.base[p] + (P)(ia.eps0 * e) * q.scl0);
        return q.base[p] + (ia.eps0 * e) * q.sclk;
    };
#pragma unroll
    for (int r = 0; r < kWR; ++r) {
        const int u = r * kWave + lane;
        const real v = val(min(t0 + u, q.N - 1));
        w.x[r] = u < nt ? v : (real)0;
    }
    const real xlv = val(max(t0 - 1, 0)), xrv = val(min(t0 + kWT, q.N - 1));
    w.xl = t0 >= 1 ? xlv : (real)0;
    w.xr = t0 + kWT < q.N ? xrv : (real)0;
}

// stores of one tile: x_i (and the noise residual), its knot bitmasks and counts
template <typename real, int MODE>
__device__ __forceinline__ void init_store(const InitSeries<real, MODE>& q, const KnotsDev<real>& kout,
                                           int gt, int lane, const InitTile<real>& w)
{
    const int t0 = (gt - q.tile0) * kWT;
    const int nt = min(kWT, q.N - t0);
#pragma unroll
    for (int r = 0; r < kWR; ++r) {
        const int u = r * kWave + lane;
        if (u < nt) {
            if (MODE == INIT_RESID ? q.out != nullptr : MODE != INIT_KNOTS) q.out[t0 + u] = w.x[r];
            if (MODE == INIT_RESID) q.resid[t0 + u] = w.x[r];
        }
    }
    int run[2] = {0, 0};
    uint64_t em[2][kWR];
    uint64_t cg = wave_ballot(w.xl > w.x[0]) & 1ull, cl = wave_ballot(w.xl < w.x[0]) & 1ull;
    const bool ends = t0 == 0 || t0 + kWT >= q.N;
#pragma unroll
    for (int r = 0; r < kWR; ++r) {
        const real rgt = r == kWR - 1 ? shift_next(w.x[r], w.xr) : row_next(w.x[r], w.x[r < kWR - 1 ? r + 1 : r]);
        row_extrema(wave_ballot(w.x[r] > rgt), wave_ballot(w.x[r] < rgt), cg, cl, em[0][r], em[1][r]);
        if (ends) {
            uint64_t valid, end;
            row_ends(t0 + r * kWave, q.N, valid, end);
#pragma unroll
            for (int ty = 0; ty < 2; ++ty) em[ty][r] = valid & (end | em[ty][r]);
        }
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) run[ty] += __popcll(em[ty][r]);
    }
    store_masks(kout.mask + 8 * (int64_t)gt, em, lane);
    if (lane == 0) {
        kout.cnt[2 * gt] = run[0];
        kout.cnt[2 * gt + 1] = run[1];
    }
}

// One wavefront per run of kInitRun consecutive tiles (grid-stride over the
// runs: the grid is capped, so any tile count fits one launch).  The series
// pointers are looked up once per run (again only where the run crosses
// into the next series), and the next tile's samples are requested before
// the current tile's stores, so each tile's loads overlap the previous
// tile's work instead of starting a chain of dependent lookups per tile.
constexpr int kInitRun = 8;

template <typename real, int MODE, bool LOOP>
__global__ __launch_bounds__(kThreads) void k_init_w(SeriesDev sd, InitArgs<real> ia, real* h_out,
                                                     KnotsDev<real> kout)
{
    constexpr int NW = kThreads / kWave;
    const int lane = threadIdx.x & 63, wv = wave_index();
    const int64_t nruns = ((int64_t)sd.ntiles + kInitRun - 1) / kInitRun;
    // one run per wavefront, or (LOOP) a grid-stride loop over the runs
    // where that grid would exceed a launch's 2^32 work-items
    for (int64_t run = (int64_t)blockIdx.x * NW + wv; run < nruns;
         run = LOOP ? run + (int64_t)gridDim.x * NW : nruns) {
        const int g0 = (int)(run * kInitRun);
        const int g1 = min(g0 + kInitRun, sd.ntiles);
        InitSeries<real, MODE> q = init_series<real, MODE>(sd, ia, h_out, sd.tile_series[g0]);
        InitTile<real> cur, nxt;
        init_load<real, MODE>(q, ia, g0, lane, cur);
        for (int gt = g0; gt < g1; ++gt) {
            InitSeries<real, MODE> qn = q;
            if (gt + 1 < g1) {
                if (gt + 1 >= q.tend) qn = init_series<real, MODE>(sd, ia, h_out, sd.tile_series[gt + 1]);
                init_load<real, MODE>(qn, ia, gt + 1, lane, nxt);
            }
            init_store<real, MODE>(q, kout, gt, lane, cur);
            cur = nxt;
            q = qn;
        }
    }
}

// ================================================================ adjoint
// With the extrema sets of every pass frozen (recorded by the forward), one
// sift pass is linear: h' = h - (U + L) / 2.  Its transpose maps the
// gradient mu of h' to that of h: mu - (G_max^T mu + G_min^T mu) / 2, where
// G^T is: per-interval moments of mu (transposed evaluation), transposed
// coefficient formulas, a solve with the transposed spline matrix (its
// interior block is the symmetric interior block of the forward matrix, so
// the forward's windowed solver is reused), transposed right-hand side and
// endpoint fix, and a scatter to the knot samples.

// 1'. Fused per-tile step for 256-sample tiles: one wavefront per tile,
// lane l owns the four consecutive samples 4l .. 4l+3.  Optionally
// mu <- broadcast, then mu <- mu - (G_max^T + G_min^T)/2 for the scatter
// pass, then the moments of mu over the knot intervals of the moment pass.
// Each lane sums its samples run by run, and the run that a lane leaves open
// is carried to the lane that ends it; the runs are put together in
// LDS and leave as contiguous 16-byte stores (written by the lanes that end
// them, 32-byte pieces at two to four places, the dense FP64 launch took 703
// us instead of 404).
// FP64 is bound by memory (samples in and out, up to 2.7 KB of moments per
// tile in the first passes: 1.6 GB), FP32 by vector instructions (438 per
// tile, 135 of the 160 us).  Densest pass of 3200 series of 16384 samples,
// FP64: 571 us with a scan keyed by run numbers and the knots found through
// LDS -> 388; 200 of 244032, FP32: 264 -> 160.

// Four consecutive values of a lane, 16 bytes per access; global memory past
// the caches (mu is read and written once per step).
template <typename real>
using Vec16 = real __attribute__((ext_vector_type(16 / sizeof(real)), aligned(sizeof(real))));
template <bool NT, typename real>
__device__ __forceinline__ void load_four(const real* p, real (&v)[4])
{
    constexpr int E = 16 / sizeof(real);
#pragma unroll
    for (int i = 0; i < 4; i += E) {
        const Vec16<real>* src = (const Vec16<real>*)(p + i);
        const Vec16<real> q = NT ? __builtin_nontemporal_load(src) : *src;
#pragma unroll
        for (int e = 0; e < E; ++e) v[i + e] = q[e];
    }
}
template <bool NT, typename real>
__device__ __forceinline__ void store_four(real* p, const real (&v)[4])
{
    constexpr int E = 16 / sizeof(real);
#pragma unroll
    for (int i = 0; i < 4; i += E) {
        Vec16<real> q;
#pragma unroll
        for (int e = 0; e < E; ++e) q[e] = v[i + e];
        if (NT) __builtin_nontemporal_store(q, (Vec16<real>*)(p + i));
        else *(Vec16<real>*)(p + i) = q;
    }
}

// One step of the segmented scan below: lanes of `take` add the values that
// the lane move CTRL brings them.
template <int CTRL, int ROWS, typename real>
__device__ __forceinline__ void open_scan_step(real (&v)[4], uint64_t take)
{
    if (take == 0ull) return;
    real w[4];
#pragma unroll
    for (int z = 0; z < 4; ++z) w[z] = dpp_row<CTRL, ROWS>(v[z], (real)0);
    if (__builtin_amdgcn_inverse_ballot_w64(take)) {
#pragma unroll
        for (int z = 0; z < 4; ++z) v[z] = v[z] + w[z];
    }
}

// Inclusive scan of the lanes' open sums: lane l ends with the sum over the
// lanes down to the nearest one that is not linked to the lane before it.
// Which lanes take part in a step is known from the mask of links by scalar
// instructions, and a step that no lane takes part in is left out (four lanes
// without a knot are rare in a dense pass).
template <typename real>
__device__ __forceinline__ void open_scan(real (&v)[4], uint64_t link)
{
    // aN: the N lanes up to this one are linked, or those of its row of 16
    const uint64_t a1 = link;
    const uint64_t a2 = a1 & ((a1 << 1) | 0x0001000100010001ull);
    const uint64_t a4 = a2 & ((a2 << 2) | 0x0003000300030003ull);
    const uint64_t a8 = a4 & ((a4 << 4) | 0x000F000F000F000Full);
    const uint64_t a16 = a8 & ((a8 << 8) | 0x00FF00FF00FF00FFull);
    open_scan_step<0x111, 0xF>(v, a1);
    open_scan_step<0x112, 0xF>(v, a2);
    open_scan_step<0x114, 0xF>(v, a4);
    open_scan_step<0x118, 0xF>(v, a8);
    open_scan_step<0x142, 0xA>(v, a16 & 0xFFFF0000FFFF0000ull);
    open_scan_step<0x143, 0xC>(v, a16 & (0x0000FFFF00000000ull | ((a16 >> 47) & 1ull ? 0xFFFFull << 48 : 0ull)));
}

// Inclusive maximum over the lanes.
__device__ __forceinline__ int max_scan(int v, int least)
{
    v = max(v, dpp_row_i<0x111, 0xF>(v, least));
    v = max(v, dpp_row_i<0x112, 0xF>(v, least));
    v = max(v, dpp_row_i<0x114, 0xF>(v, least));
    v = max(v, dpp_row_i<0x118, 0xF>(v, least));
    v = max(v, dpp_row_i<0x142, 0xA>(v, least));
    return max(v, dpp_row_i<0x143, 0xC>(v, least));
}

constexpr int kAdjKC = kWT / 2 + 2;   // knots of one type in a tile, at most

template <typename real>
__device__ __forceinline__ void adj_tile(const AdjTileArgs<real>& a, int gt, int lane, real* sm)
{
    const SeriesDev& sd = a.sd;
    const int s = load_scalar(sd.tile_series + gt);
    const int t0 = (gt - load_scalar(sd.tile0 + s)) * kWT;
    const int nt = min(kWT, load_scalar(sd.len + s) - t0);
    const int64_t kb = load_scalar(sd.kbase + s);
    real* mu = a.mu + load_scalar(sd.off + s) + t0;
    const int ub = 4 * lane;

    real v[4];
    bool dirty = false;
    {
        const real* src = mu;
        if (a.bcast) {
            src = a.bcast + load_scalar(a.chan_off + load_scalar(sd.chan + s)) + t0;
            dirty = true;
        }
        if (nt == kWT) {
            load_four<true>(src + ub, v);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = ub + q < nt ? src[ub + q] : (real)0;
        }
    }
    // ---- scatter of the knot gradients of pass sc: a sample that is a knot
    // adds the gradient of that knot
    if (a.sc.mask && load_scalar(a.sc.n + 2 * s) > 3 && load_scalar(a.sc.n + 2 * s + 1) > 3) {
        real g[2][4];
#pragma unroll
        for (int ty = 0; ty < 2; ++ty) {
            uint64_t bm[4];
            quad_masks(quad_byte(a.sc.mask, gt, ty, lane), lane, bm);
            const real* ga = a.ga + kb + (ty ? sd.kstride : 0) + load_scalar(a.sc.pre + 2 * gt + ty);
            unsigned r = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) r = rank_below(bm[q], r);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                g[ty][q] = (real)0;
                if (__builtin_amdgcn_inverse_ballot_w64(bm[q])) g[ty][q] = ga[r];
                r = add_bit(r, bm[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = v[q] - (g[0][q] + g[1][q]) / (real)2;
        dirty = true;
    }
    if (dirty) {
        if (nt == kWT) {
            store_four<true>(mu + ub, v);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (ub + q < nt) mu[ub + q] = v[q];
        }
    }
    // ---- moments of mu over the intervals of pass mo: run r of the tile are
    // the samples after its knot r - 1 up to its knot r (sample 0 of the
    // series joins run 1, the interval (x_0, x_1]), and t is the distance
    // from the knot before
    if (!(a.mo.mask && load_scalar(a.mo.n + 2 * s) > 3 && load_scalar(a.mo.n + 2 * s + 1) > 3)) return;
#pragma unroll
    for (int ty = 0; ty < 2; ++ty) {
        const int cnt = load_scalar(a.mo.cnt + 2 * gt + ty), pre = load_scalar(a.mo.pre + 2 * gt + ty);
        // the knot before the tile, from its first sample (0 where sample 0
        // of the series is the first knot)
        const int left = t0 > 0 ? load_scalar(a.mo.left + 2 * gt + ty) - t0 : 0;
        uint64_t bm[4];
        quad_masks(quad_byte(a.mo.mask, gt, ty, lane), lane, bm);
        if (t0 == 0) bm[0] &= ~1ull;
        real* e = a.edge + 4 * (4 * (int64_t)gt + 2 * ty);
        real* mom = a.mom + 4 * (kb + (ty ? sd.kstride : 0) + pre - 1);
        // distance of the lane's samples from the knot before them
        int t[4];
        {
            int last = left;
#pragma unroll
            for (int q = 0; q < 4; ++q) last = __builtin_amdgcn_inverse_ballot_w64(bm[q]) ? ub + q : last;
            t[0] = ub - dpp_prev_i(max_scan(last, left), left);
#pragma unroll
            for (int q = 0; q < 3; ++q) t[q + 1] = __builtin_amdgcn_inverse_ballot_w64(bm[q]) ? 1 : t[q] + 1;
        }
        // moments of the runs within the lane; one that ends on its last
        // sample (or goes on) is open
        real run[4] = {(real)0, (real)0, (real)0, (real)0};
        int r = t0 == 0 ? 1 : 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) r = rank_below(bm[q], r);
        real* mine = &sm[4 * r];
        real* d = mine;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            real m = v[q];
            run[0] = run[0] + m;
#pragma unroll
            for (int z = 1; z < 4; ++z) {
                m = m * (real)t[q];
                run[z] = run[z] + m;
            }
            if (q < 3 && __builtin_amdgcn_inverse_ballot_w64(bm[q])) {
                store_four<false>(d, run);
                d += 4;
#pragma unroll
                for (int z = 0; z < 4; ++z) run[z] = (real)0;
            }
        }
        const uint64_t inside = bm[0] | bm[1] | bm[2], after = bm[3] << 1;
        open_scan(run, ~(inside | after));
        if (__builtin_amdgcn_inverse_ballot_w64(bm[3])) store_four<false>(d, run);
        if (lane == kWave - 1) {
            real rest[4];
#pragma unroll
            for (int z = 0; z < 4; ++z) rest[z] = bm[3] >> 63 ? (real)0 : run[z];
            store_four<false>(e + (cnt > 0 ? 4 : 0), rest);
        }
        // the first run that ends inside the lane goes on from the lane before
#pragma unroll
        for (int z = 0; z < 4; ++z) run[z] = shift_prev(run[z], (real)0);
        if (__builtin_amdgcn_inverse_ballot_w64(inside & ~after)) {
            real m[4];
            load_four<false>(mine, m);
#pragma unroll
            for (int z = 0; z < 4; ++z) m[z] = run[z] + m[z];
            store_four<false>(mine, m);
        }
        wave_sync();
        // runs 1 .. cnt - 1 lie side by side in mom, run 0 goes to the edge
        constexpr int E = 16 / sizeof(real);
        for (int i = E * lane; i < 4 * cnt; i += E * kWave)
            *(Vec16<real>*)(i < 4 ? e + i : mom + i) = *(const Vec16<real>*)&sm[i];
        wave_sync();
    }
}

// One wavefront per tile (LOOP = false), or a grid-stride loop over the
// tiles where one wave per tile would exceed a launch's 2^32 work-items.
template <typename real, bool LOOP>
__global__ __launch_bounds__(kThreads) void k_adj_tile(AdjTileArgs<real> a)
{
    constexpr int NW = kThreads / kWave;
    __shared__ alignas(16) real s_mom[NW][4 * kAdjKC];
    const int lane = threadIdx.x & 63, wv = wave_index();
    if (!LOOP) {
        const int gt = blockIdx.x * NW + wv;
        if (gt < a.sd.ntiles) adj_tile<real>(a, gt, lane, s_mom[wv]);
        return;
    }
    for (int gt = blockIdx.x * NW + wv; gt < a.sd.ntiles; gt += gridDim.x * NW)
        adj_tile<real>(a, gt, lane, s_mom[wv]);
}

// 2. intervals that leave their tile: the last run of the tile holding the
// left knot plus the first runs of the following tiles up to the right knot
template <typename real>
__global__ void k_adj_span(AdjArgs<real> a)
{
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    const SeriesDev& sd = a.sd;
    if (gt >= sd.ntiles) return;
    const int s = sd.tile_series[gt];
    const int n0 = a.ps.n[2 * s], n1 = a.ps.n[2 * s + 1];
    if (!(n0 > 3 && n1 > 3)) return;
    for (int ty = 0; ty < 2; ++ty) {
        const int cnt = a.ps.cnt[2 * gt + ty];
        if (cnt == 0) continue;
        const int g = a.ps.pre[2 * gt + ty] + cnt - 1;
        if (g >= (ty ? n1 : n0) - 1) continue;
        const real* e = a.edge + 4 * (4 * (int64_t)gt + 2 * ty + 1);
        real m0 = e[0], m1 = e[1], m2 = e[2], m3 = e[3];
        // up to the tile holding the next knot (known from the record, so
        // the loads do not wait on each other)
        const int last = sd.tile0[s] + a.ps.right[2 * gt + ty] / kWT;
        int tau = gt + 1;
        // eight tiles at a time: all loads first, then the adds in order
        for (; tau + 7 <= last; tau += 8) {
            real f[8][4];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const real* fp = a.edge + 4 * (4 * (int64_t)(tau + u) + 2 * ty);
#pragma unroll
                for (int m = 0; m < 4; ++m) f[u][m] = fp[m];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                m0 += f[u][0];
                m1 += f[u][1];
                m2 += f[u][2];
                m3 += f[u][3];
            }
        }
        for (; tau <= last; ++tau) {
            const real* f = a.edge + 4 * (4 * (int64_t)tau + 2 * ty);
            m0 += f[0];
            m1 += f[1];
            m2 += f[2];
            m3 += f[3];
        }
        real* dst = a.mom + 4 * (sd.kbase[s] + (ty ? sd.kstride : 0) + g);
        dst[0] = m0;
        dst[1] = m1;
        dst[2] = m2;
        dst[3] = m3;
    }
}

// 3. knot gradients: right-hand side gc of the transposed solve from the
// moments (transposed coefficient formulas, cudaICEEMDAN.cu:394-398), the
// solve, the transposed right-hand side f(a) (:333-341) and endpoint fix
// (:209-291).  One wavefront per window, the forward's window geometry.
// (three waves per SIMD: the compiler is held to 168 registers)
template <typename real, int B, int H>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_adj_knot(AdjArgs<real> a)
{
    constexpr int W = kWave * B;
    constexpr int K = W - 2 * H;
    constexpr int NW = kThreads / kWave;
    __shared__ real s_f[NW][W];            // knot-value gradients of the window rows
    __shared__ int s_pos[NW][W + 2];       // knot positions g0-1 .. g0+W
    __shared__ int s_tpre[NW][kWave];
    __shared__ uint64_t s_tmask[NW][kWave][kTMaskW];
    const int wv = wave_index(), lane = threadIdx.x & 63;
    real* sf = s_f[wv];
    int* sp = s_pos[wv];
    const real third = (real)1 / (real)3;
    // window items and series metadata through the scalar cache (read-only here)
    const unsigned total = load_scalar(a.wincount);
    for (unsigned item = blockIdx.x * NW + wv; item < total; item += gridDim.x * NW) {
        const int s = load_scalar(a.winlist + kWinItem * item);
        const int code = load_scalar(a.winlist + kWinItem * item + 1);
        const int hint = load_scalar(a.winlist + kWinItem * item + 2);
        const int type = code & 1;
        const int w = code >> 1;
        const int n0 = load_scalar(a.ps.n + 2 * s), n1 = load_scalar(a.ps.n + 2 * s + 1);
        if (!(n0 > 3 && n1 > 3)) continue;
        const int n = type ? n1 : n0;
        const int64_t kb = load_scalar(a.sd.kbase + s) + (type ? a.sd.kstride : 0);
        const long g0 = (long)w * K - H;
        // knot positions of the window (and one beyond each side) from the
        // pass's bitmasks: sp index = g - lo
        const long lo = g0 - 1;
        const int glo = (int)max(lo, 0L);
        const int ghi = (int)min(lo + W + 2, (long)n);
        gather_positions<kTMaskW>(a.sd, a.ps.mask, a.ps.pre, a.ps.cnt, s, type, lo, glo, ghi, sp,
                                  s_tpre[wv], s_tmask[wv], hint, n);
        wave_sync();
        // lane l owns window rows r = l*B + q (knot gb + q); everything a row
        // needs comes from its own lane's registers or a neighbour lane's
        const long gb = g0 + (long)lane * B;
        // positions of knots gb-1 .. gb+B (xk[j] <-> knot gb-1+j), clamped
        // into the series (values past its ends are never used)
        int xk[B + 2];
#pragma unroll
        for (int j = 0; j < B + 2; ++j) {
            const long g = gb - 1 + j;
            xk[j] = sp[min(max(g, 0L), (long)n - 1) - lo];
        }
        // interval gb-1+j (j = 0..B): its moments feed its left knot (row j-1)
        // and its right knot (row j) through the transposed coefficient
        // formulas (cudaICEEMDAN.cu:394-398).  gc = right-hand side of the
        // transposed solve, vp = the part of the knot gradient without the
        // solution; ih = reciprocal interval length.  (The adjoint is compared
        // to tolerance, not bit for bit: one reciprocal per interval.)
        real gc[B], vp[B], ih[B + 1];
        real gr_prev = (real)0, vr_prev = (real)0;
#pragma unroll
        for (int j = 0; j <= B; ++j) {
            const long gg = gb - 1 + j;
            const bool in = gg >= 0 && gg <= n - 2;
            const real* m = a.mom + 4 * (kb + (in ? gg : 0));
            const real m0 = m[0], m1 = m[1], m2 = m[2], m3 = m[3];
            const real h = (real)(xk[j + 1] - xk[j]);
            const real ihh = in ? (real)1 / h : (real)0;
            ih[j] = ihh;
            const real gl = in ? m2 - (real)2 * third * h * m1 - m3 * ihh * third : (real)0;
            const real gr = in ? m3 * ihh * third - h * third * m1 : (real)0;
            const real vl = in ? m0 - m1 * ihh : (real)0;
            const real vr = in ? m1 * ihh : (real)0;
            if (j >= 1) {
                const int q = j - 1;
                const long g = gb + q;
                gc[q] = (g >= 1 && g <= n - 2) ? gl + gr_prev : (real)0;
                vp[q] = vl + vr_prev;
            }
            gr_prev = gr;
            vr_prev = vr;
        }
        real xs[B];
        partition_pcr<real, B, true>(
            lane,
            [&](int q, real& dl, real& d, real& du, real& f) {
                const long g = gb + q;
                if (g <= 0 || g >= n - 1) {
                    dl = (real)0; d = (real)1; du = (real)0; f = (real)0;
                    return;
                }
                const int hl = xk[q + 1] - xk[q];
                const int hr = xk[q + 2] - xk[q + 1];
                dl = (real)hl;
                du = (real)hr;
                d = (real)(2 * (hl + hr));
                f = gc[q];
            },
            xs);
        // solution of the rows just outside this lane's block
        const real xprev = shift_prev(xs[B - 1], (real)0);
        const real xnext = shift_next(xs[0], (real)0);
        // base knot gradient of every row with both neighbours in the window
#pragma unroll
        for (int q = 0; q < B; ++q) {
            const int r = lane * B + q;
            const long g = gb + q;
            real v = (real)0;
            if (g >= 0 && g < n && r >= 1 && r <= W - 2) {
                const real sm1 = q == 0 ? xprev : xs[q > 0 ? q - 1 : 0];
                const real sp1 = q == B - 1 ? xnext : xs[q < B - 1 ? q + 1 : q];
                v = vp[q];
                if (g - 1 >= 1 && g - 1 <= n - 2) v = v + (real)3 * sm1 * ih[q];
                if (g >= 1 && g <= n - 2) v = v - (real)3 * xs[q] * (ih[q + 1] + ih[q]);
                if (g + 1 >= 1 && g + 1 <= n - 2) v = v + (real)3 * sp1 * ih[q + 1];
            }
            sf[r] = v;
        }
        wave_sync();
        // endpoint fix: a_0 = a_1 (1 + rho) - a_2 rho when it replaced a_0
        if (lane == 0 && n >= 6) {
            const int* xp = sp - lo;   // xp[g] = position of knot g (g in the window)
            const long r0 = 0 - g0;
            if (r0 >= 1 && r0 + 2 <= W - 2 && a.ps.fixf[4 * s + 2 * type]) {
                const real rho = (real)(xp[1] - xp[0]) / (real)(xp[2] - xp[1]);
                sf[r0 + 1] = sf[r0 + 1] + sf[r0] * ((real)1 + rho);
                sf[r0 + 2] = sf[r0 + 2] - sf[r0] * rho;
                sf[r0] = (real)0;
            }
            const long r1 = (long)(n - 1) - g0;
            if (r1 - 2 >= 1 && r1 <= W - 2 && a.ps.fixf[4 * s + 2 * type + 1]) {
                const real rho = (real)(xp[n - 1] - xp[n - 2]) / (real)(xp[n - 2] - xp[n - 3]);
                sf[r1 - 1] = sf[r1 - 1] + sf[r1] * ((real)1 + rho);
                sf[r1 - 2] = sf[r1 - 2] - sf[r1] * rho;
                sf[r1] = (real)0;
            }
        }
        wave_sync();
        for (int r = H + lane; r < H + K; r += kWave) {
            const long g = g0 + r;
            if (g < n) a.ga[kb + g] = sf[r];
        }
        wave_sync();
    }
}

template <typename real>
__global__ void k_adj_seed(const real* gimf, int M, int N, int64_t stride, real* gr)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    gr[p] = gimf[p];
    for (int k = 1; k < M; ++k)
        gr[(int64_t)k * stride + p] = gimf[(int64_t)k * N + p] - gimf[(int64_t)(k - 1) * N + p];
}

// Realizations whose samples are requested before the first is added, in the
// sums over i (one at a time, a channel of 4096 samples and 50 realizations
// took 21 us).
constexpr int kEnsAhead = 8;

// stage level: mu of every realization starts as dL/dr_{k+1} of its channel
// g_x_i = (lambda - mu_i) / I; gacc = sum_i g_x_i (sequential in i)
template <typename real>
__global__ void k_adj_accum(int I, const int* chan_len, const int64_t* chan_off, SeriesDev sd,
                            const real* gr_next, const real* mu, real* gacc)
{
    const int c = blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const int N = chan_len[c];
    if (p >= N) return;
    const real lam = gr_next[chan_off[c] + p];
    // the channel's series lie back to back
    const real* m = mu + sd.off[c * I] + p;
    real acc = (real)0;
    int i = 0;
    for (; i + kEnsAhead <= I; i += kEnsAhead) {
        real v[kEnsAhead];
#pragma unroll
        for (int q = 0; q < kEnsAhead; ++q) v[q] = m[(int64_t)(i + q) * N];
#pragma unroll
        for (int q = 0; q < kEnsAhead; ++q) acc = acc + (lam - v[q]) / (real)I;
    }
    for (; i < I; ++i) acc = acc + (lam - m[(int64_t)i * N]) / (real)I;
    gacc[chan_off[c] + p] = acc;
}

// dots[s] = <g_x_s, E_s> (canonical order), one workgroup per series
template <typename real>
__global__ __launch_bounds__(1024) void k_adj_dot(int I, SeriesDev sd, const int64_t* chan_off,
                                                  const real* gr_next, const real* mu,
                                                  const real* E, real* dots)
{
    __shared__ real sred[1024];
    const int s = blockIdx.x;
    const int N = sd.len[s];
    const real* lam = gr_next + chan_off[sd.chan[s]];
    const real* m = mu + sd.off[s];
    const real* e = E + sd.eoff[s];
    struct T3 { real l, m, e; };
    const real acc = canon_lane_sum<real>(
        N, [&](int p) { return T3{lam[p], m[p], e[p]}; },
        [&](const T3& t) { return ((t.l - t.m) / (real)I) * t.e; });
    const real d = canon_sum_block<real>(acc, sred);
    if (threadIdx.x == 0) dots[s] = d;
}

// coef[c] = eps0 sum_i dots / ((N - 1) std(r_k)) (sequential in i), one wave
// per channel
template <typename real>
__global__ __launch_bounds__(kWave) void k_adj_coef(int I, const int* chan_len, const real* dots,
                                                    const double* sq, real eps0, real* coef)
{
    const int c = blockIdx.x, lane = threadIdx.x;
    real dsum = (real)0;
    for (int i0 = 0; i0 < I; i0 += kWave) {
        const real v = i0 + lane < I ? dots[c * I + i0 + lane] : (real)0;
        const int m = min(kWave, I - i0);
        for (int l = 0; l < m; ++l) dsum = dsum + lane_value(v, l);
    }
    if (lane == 0) coef[c] = eps0 * dsum / ((real)(chan_len[c] - 1) * (real)sq[c]);
}

// gr_k += gacc (+ coef (r_k - mean(r_k)), k >= 1: coef is null at stage 0)
template <typename real>
__global__ void k_adj_stage(const int* chan_len, const int64_t* chan_off, const real* gacc,
                            const real* coef, const real* mean, const real* r_k, real* gr_k)
{
    const int c = blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= chan_len[c]) return;
    const int64_t o = chan_off[c] + p;
    real v = gr_k[o] + gacc[o];
    if (coef) v = v + coef[c] * (r_k[o] - mean[c]);
    gr_k[o] = v;
}

// dL/dy from dL/dx~ with x~ = y / std(y)
template <typename real>
__global__ __launch_bounds__(1024) void k_adj_input(const int* chan_len, const int64_t* chan_off,
                                                    const real* y, const real* gxt, real* gy)
{
    __shared__ real sred[1024];
    const int c = blockIdx.x;
    const int N = chan_len[c];
    const int64_t o = chan_off[c];
    auto at = [&](int p) { return y[o + p]; };
    const real mu = canon_sum_block<real>(canon_lane_sum<real>(N, at, [](real v) { return v; }), sred) *
                    (real)(1.0 / (double)N);
    const real var = canon_sum_block<real>(canon_lane_sum<real>(N, at, [&](real v) {
                                               const real dv = v - mu;
                                               return dv * dv;
                                           }), sred) * (real)(1.0 / (double)(N - 1));
    struct T2 { real g, y; };
    const real dot = canon_sum_block<real>(
        canon_lane_sum<real>(N, [&](int p) { return T2{gxt[o + p], y[o + p]}; },
                             [](const T2& t) { return t.g * t.y; }), sred);
    const real sx = (real)1 / sqrt(var);
    for (int p = threadIdx.x; p < N; p += 1024)
        gy[o + p] = sx * gxt[o + p] - sx * sx * sx * dot * (y[o + p] - mu) / (real)(N - 1);
}

// --------------------------------------------------------------------- noise

// value (i, p): Philox4x64-10 block q = p/4, counter (q, i, 0, 0), key (seed, 0);
// u = ((bits >> 11) + 0.5) * 2^-53; Box-Muller on (u0,u1) and (u2,u3).
// One launch for the rows of several lengths: length blockIdx.z of `len`
// (its rows from row_off[z]), or the one length N.
template <typename real>
__global__ void k_noise(uint64_t seed, const int* len, const int64_t* row_off, int64_t N, real* out)
{
    const int i = blockIdx.y;
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (len) N = len[blockIdx.z];
    if (4 * q >= N) return;
    const u64x4 b = philox4x64_10((uint64_t)q, (uint64_t)i, 0, 0, seed, 0);
    const double TWO_PI = 6.283185307179586476925286766559;
    double u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) u[j] = ((double)(b.v[j] >> 11) + 0.5) * 0x1.0p-53;
    const double r0 = sqrt(-2.0 * log(u[0]));
    const double r1 = sqrt(-2.0 * log(u[2]));
    double z[4];
    z[0] = r0 * cos(TWO_PI * u[1]);
    z[1] = r0 * sin(TWO_PI * u[1]);
    z[2] = r1 * cos(TWO_PI * u[3]);
    z[3] = r1 * sin(TWO_PI * u[3]);
    real* row = out + (row_off ? row_off[blockIdx.z] : 0) + (int64_t)i * N;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (4 * q + j < N) row[4 * q + j] = (real)z[j];
}

// ------------------------------------------------------------ stage kernels

// ensemble mean of x_i - h_i over realizations, sequential in i
// (produceFirstIMF :41-55, produceResidue + averageUpdateSignal :582-607)
template <typename real>
__device__ __forceinline__ real acc_stage0(real tem, double invI, real d)
{
    return (real)((double)tem + invI * (double)d);
}

// The loads of kEnsAhead realizations go out before the first is added.
template <typename real, bool STAGE0>
__global__ void k_ensemble(EnsembleArgs<real> a)
{
    using P = typename Promote<real>::type;
    const int c = blockIdx.y;
    const int N = a.chan_len[c];
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const int I = a.I;
    const int64_t co = a.chan_off[c];
    // row `stage` of channel c's [M][N] output
    real* imf_k = a.imf + a.chan_imf_off[c] + (int64_t)a.stage * N;
    // the channel's series and its noise rows lie back to back
    const int s0 = c * I;
    const int64_t ho = a.ser_off[s0] + p;
    const real* hs[2] = {a.hA + ho, a.hB + ho};
    const real* e = a.E + a.ser_eoff[s0] + p;
    const int n0 = a.ser_nidx[s0];
    const real base = STAGE0 ? a.xt[co + p] : a.r[co + p];
    const double invI = 1.0 / (double)I;
    const real sqc = STAGE0 ? (real)0 : (real)a.sq[c];
    real tem = (real)0;
    auto add = [&](int i, real hv, real ev) {
        if (STAGE0) {
            const real x = (real)((P)base + (P)(a.eps0 * ev) * (P)a.inv[n0 + i]);
            tem = acc_stage0<real>(tem, invI, x - hv);
        } else {
            const real x = base + (a.eps0 * ev) * sqc;
            tem = tem + (x - hv);
        }
    };
    int i = 0;
    for (; i + kEnsAhead <= I; i += kEnsAhead) {
        real hv[kEnsAhead], ev[kEnsAhead];
#pragma unroll
        for (int q = 0; q < kEnsAhead; ++q) {
            const int par = a.mode_parity ? (a.mode_parity[s0 + i + q] & 1) : a.fixed_parity;
            hv[q] = (par ? hs[1] : hs[0])[(int64_t)(i + q) * N];
            ev[q] = e[(int64_t)(i + q) * N];
        }
#pragma unroll
        for (int q = 0; q < kEnsAhead; ++q) add(i + q, hv[q], ev[q]);
    }
    for (; i < I; ++i) {
        const int par = a.mode_parity ? (a.mode_parity[s0 + i] & 1) : a.fixed_parity;
        add(i, (par ? hs[1] : hs[0])[(int64_t)i * N], e[(int64_t)i * N]);
    }
    const real rn = STAGE0 ? tem : tem / (real)I;
    imf_k[p] = base - rn;
    a.r[co + p] = rn;
    if (a.r_next) a.r_next[co + p] = rn;
    // the last stage's residue is row M - 1 (cudaICEEMDAN.cu:1298)
    if (a.last) imf_k[N + p] = rn;
}

// x~ = y * (1 / sqrt(var(y)))  (standardizeRunning, cudaICEEMDAN.cu:57-66)
template <typename real>
__global__ void k_standardize(const real* y, const real* var, real* xt, const int* chan_len,
                              const int64_t* chan_off)
{
    using P = typename Promote<real>::type;
    const int c = blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= chan_len[c]) return;
    const P inv = 1.0 / (P)sqrt(var[c]);
    const int64_t o = chan_off[c] + p;
    xt[o] = (real)((P)y[o] * inv);
}

// Caller buffers of up to kPtrBatch channels to (IN) or from the plan's:
// channel c0 + blockIdx.y, rows * chan_len elements
template <typename real, bool IN>
__global__ void k_channels(PtrBatch ptr, int c0, int rows, const int* chan_len, const int64_t* off,
                           real* own)
{
    const int c = c0 + blockIdx.y;
    const int64_t n = (int64_t)rows * chan_len[c];
    real* q = own + off[c];
    real* u = (real*)ptr.p[blockIdx.y];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        if (IN) q[i] = u[i];
        else u[i] = q[i];
    }
}

// elementwise kernels: grid-stride with 64-bit indices (capped grids)
template <typename real>
__global__ void k_copy(real* dst, const real* src, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// dst[s] = (parity[s] odd ? hB : hA)[s] for every series (RILLING export)
template <typename real>
__global__ void k_select_copy(SeriesDev sd, const real* hA, const real* hB, const int* parity,
                              real* dst)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    for (int s = blockIdx.y; s < sd.nseries; s += gridDim.y) {
        if (p >= sd.len[s]) continue;
        const int64_t o = sd.off[s] + p;
        dst[o] = ((parity[s] & 1) ? hB : hA)[o];
    }
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Order-independent 64-bit digest of the knot sets of a pass input, per
// series: the sum (mod 2^64) over the series' tiles of a mix of each of the
// tile's eight bitmask words with its (tile, type, row) index.  Two passes
// with equal digests met the same knot sets (up to a hash collision).
__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    // splitmix64 finalizer (Steele, Lea, Flood 2014)
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void k_knot_digest(const int* tile_series, const int* tile0, const uint64_t* mask,
                              int ntiles, unsigned long long* out)
{
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    if (gt >= ntiles) return;
    const int s = tile_series[gt];
    const uint64_t t = (uint64_t)(gt - tile0[s]);
    uint64_t h = 0;
#pragma unroll
    for (int q = 0; q < 2 * kWR; ++q) h += mix64(mask[8 * (int64_t)gt + q] ^ mix64(8 * t + q + 1));
    atomicAdd(out + s, (unsigned long long)h);
}

__global__ void k_check_index(const int* x, int64_t N, int* err)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N && x[i] != (int)i) atomicOr(err, ICM_DEVERR_INDEX);
}

// ---------------------------------------------------------------- launchers

static inline unsigned blocks_for(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }
// grid of a grid-stride launch: at most 2^20 workgroups (2^28 work-items)
static inline unsigned capped_blocks(int64_t n, int b)
{
    const int64_t g = (n + b - 1) / b;
    return (unsigned)(g < 1 ? 1 : (g > (1 << 20) ? (1 << 20) : g));
}
// workgroups of kThreads for n items, b per workgroup, if that grid fits one
// launch (fewer than 2^32 work-items); else 0 (the grid-stride instance)
static inline unsigned full_blocks(int64_t n, int b)
{
    const int64_t g = std::max<int64_t>(1, (n + b - 1) / b);
    return g * kThreads < ((int64_t)1 << 32) ? (unsigned)g : 0u;
}

// Workgroups of `kernel` (kThreads each) that the device keeps resident at
// once, per device (the grid of a persistent launch).
template <typename K>
static int resident_groups(K kernel)
{
    static std::mutex mu;
    static std::map<std::pair<const void*, int>, int> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    const auto key = std::make_pair((const void*)kernel, dev);
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, kThreads, 0) != hipSuccess ||
        per <= 0)
        per = 4;
    cache[key] = cus * per;
    return cus * per;
}

// tile size (samples per tile) is a plan parameter: sd.cap = T/2 + 2
template <typename real, int MODE>
static void launch_init_mode(bool loop, dim3 grid, hipStream_t st, const SeriesDev& sd,
                             const InitArgs<real>& ia, real* h_out, const KnotsDev<real>& kout)
{
    if (loop)
        hipLaunchKernelGGL((k_init_w<real, MODE, true>), grid, dim3(kThreads), 0, st, sd, ia, h_out,
                           kout);
    else
        hipLaunchKernelGGL((k_init_w<real, MODE, false>), grid, dim3(kThreads), 0, st, sd, ia, h_out,
                           kout);
}

template <typename real>
hipError_t launch_init(const SeriesDev& sd, const InitArgs<real>& ia, real* h_out,
                       const KnotsDev<real>& kout, const PassCtl&, hipStream_t st, bool force_loop)
{
    const int64_t runs = ((int64_t)sd.ntiles + kInitRun - 1) / kInitRun;
    const unsigned full = force_loop ? 0u : full_blocks(runs, kThreads / kWave);
    const bool loop = full == 0;
    const dim3 grid(loop ? capped_blocks(runs, kThreads / kWave) : full);
    switch (ia.mode) {
    case INIT_COPY: launch_init_mode<real, INIT_COPY>(loop, grid, st, sd, ia, h_out, kout); break;
    case INIT_RESID: launch_init_mode<real, INIT_RESID>(loop, grid, st, sd, ia, h_out, kout); break;
    case INIT_STAGE0: launch_init_mode<real, INIT_STAGE0>(loop, grid, st, sd, ia, h_out, kout); break;
    case INIT_KNOTS: launch_init_mode<real, INIT_KNOTS>(loop, grid, st, sd, ia, h_out, kout); break;
    default: launch_init_mode<real, INIT_STAGEK>(loop, grid, st, sd, ia, h_out, kout); break;
    }
    return hipGetLastError();
}

template <typename real>
hipError_t launch_knot_prefix(const SeriesDev& sd, const KnotsDev<real>& k, const real* h,
                              const PassCtl& pc, const int* active, hipStream_t st)
{
    if (sd.max_tiles <= kPWTiles)
        hipLaunchKernelGGL((k_knot_prefix_w<real>), dim3(blocks_for(sd.nseries, kThreads / kWave)),
                           dim3(kThreads), 0, st, sd, k, h, pc, active);
    else if (sd.max_tiles <= kPT)
        hipLaunchKernelGGL((k_knot_prefix_1<real>), dim3(sd.nseries), dim3(kPT), 0, st, sd, k, h,
                           pc, active);
    else
        hipLaunchKernelGGL((k_knot_prefix_b<real>), dim3(sd.nseries), dim3(kPT), 0, st, sd, k, h,
                           pc, active);
    return hipGetLastError();
}

// grid of a k_sift_w launch: with a work queue, what the device keeps
// resident (no more than one wave per segment); without, one wave per segment
template <typename K>
static dim3 sift_grid(K kernel, const unsigned* queue, int nsegs)
{
    const int64_t need = blocks_for(nsegs, kThreads / kWave);
    if (!queue) return dim3((unsigned)need);
    return dim3((unsigned)std::max<int64_t>(1, std::min<int64_t>(need, resident_groups(kernel))));
}

template <typename real, bool RILL, int KC, bool NT>
static void launch_sift_w(const SiftArgs<real>& a, int nsegs, hipStream_t st)
{
    if (a.queue) {
        // (past 2^32 work-items the samples never fit the caches)
        auto k = k_sift_w<real, RILL, KC, true, true>;
        hipLaunchKernelGGL(k, sift_grid(k, a.queue, nsegs), dim3(kThreads), 0, st, a, nsegs);
    } else {
        auto k = k_sift_w<real, RILL, KC, NT, false>;
        hipLaunchKernelGGL(k, sift_grid(k, a.queue, nsegs), dim3(kThreads), 0, st, a, nsegs);
    }
}

template <typename real, bool RILL, bool NT>
static hipError_t launch_sift_as(const SiftArgs<real>& a, int nsegs, hipStream_t st)
{
    if (!a.ovf_segs) {
        launch_sift_w<real, RILL, kWKC, NT>(a, nsegs, st);
        return hipGetLastError();
    }
    // sparse pass: if few tiles of the input overflow the small knot tables
    // (the knot prefix counted them), small tables (more waves per SIMD) and
    // then the listed overflow tiles with full tables; else the small-table
    // launch returns at once and the second launch sifts every segment.
    // Its grid is what the full-table kernel keeps resident (four
    // workgroups per CU), so it costs little when it has nothing to do.
    const dim3 lgrid(std::min<unsigned>(blocks_for(nsegs, kThreads / kWave), 1024u));
    launch_sift_w<real, RILL, kWKS, NT>(a, nsegs, st);
    hipLaunchKernelGGL((k_sift_list<real, RILL, NT>), lgrid, dim3(kThreads), 0, st, a, nsegs);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_sift(const SiftArgs<real>& a, int nsegs, hipStream_t st)
{
    if (a.sx_cnt)
        return a.past_caches ? launch_sift_as<real, true, true>(a, nsegs, st)
                             : launch_sift_as<real, true, false>(a, nsegs, st);
    return a.past_caches ? launch_sift_as<real, false, true>(a, nsegs, st)
                         : launch_sift_as<real, false, false>(a, nsegs, st);
}

template <typename real>
hipError_t launch_solve(const SolveArgs<real>& a, int grid, hipStream_t st)
{
    if (a.nak)
        hipLaunchKernelGGL((k_solve<real, Geom<real>::B, Geom<real>::H, true>), dim3(grid),
                           dim3(kThreads), 0, st, a);
    else
        hipLaunchKernelGGL((k_solve<real, Geom<real>::B, Geom<real>::H, false>), dim3(grid),
                           dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_rilling_decide(const SeriesDev& sd, const int* nk, const int* sx_cnt,
                                 const int* sx_mark, int* active, int* stop_pass, int* subs,
                                 int pass, int cap, const unsigned* run, unsigned* n_active,
                                 hipStream_t st)
{
    hipLaunchKernelGGL((k_rilling_decide<real>), dim3(sd.nseries), dim3(kWave), 0, st, sd, nk,
                       sx_cnt, sx_mark, active, stop_pass, subs, pass, cap, run, n_active);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_series_var(const real* base, const int64_t* off, int64_t stride, const int* len,
                             int nser, real* var_out, real* mean_out, double* scale_out, int scale,
                             hipStream_t st)
{
    hipLaunchKernelGGL((k_series_var<real>), dim3(nser), dim3(1024), 0, st, base, off, stride, len,
                       var_out, mean_out, scale_out, scale);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_noise(uint64_t seed, int I, int64_t N, real* out, hipStream_t st)
{
    const int64_t nq = (N + 3) / 4;
    hipLaunchKernelGGL((k_noise<real>), dim3(blocks_for(nq, 256), I), dim3(256), 0, st, seed,
                       (const int*)nullptr, (const int64_t*)nullptr, N, out);
    return hipGetLastError();
}

// The lengths host_len[0 .. ngroups), also at `len` on the device, in their
// order: as many per launch as leave at least half of its workgroups with
// samples (each length takes the grid of the longest), below 2^31 work-items.
// 1000 lengths of 256 samples and up behind one of 2^20, I = 50,
// FP32, per forward: all in one grid 11.3 ms, a launch per length 4.4, these two
// launches 0.75.
template <typename real>
hipError_t launch_noise_groups(uint64_t seed, int I, int ngroups, const int64_t* host_len, const int* len,
                               const int64_t* row_off, real* out, hipStream_t st)
{
    for (int g = 0, n = 0; g < ngroups; g += n) {
        int64_t longest = 0, sum = 0;
        for (n = 0; g + n < ngroups && n < 65535; ++n) {
            const int64_t b = blocks_for((host_len[g + n] + 3) / 4, 256), m = std::max(longest, b);
            if (n > 0 && (m * (n + 1) > 2 * (sum + b) || m * (n + 1) * 256 * I > (int64_t)1 << 31)) break;
            longest = m;
            sum += b;
        }
        hipLaunchKernelGGL((k_noise<real>), dim3((unsigned)longest, I, n), dim3(256), 0, st, seed, len + g,
                           row_off + g, (int64_t)0, out);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <typename real>
hipError_t launch_ensemble(const EnsembleArgs<real>& a, int nchan, int max_len, hipStream_t st)
{
    const dim3 g(blocks_for(max_len, 256), nchan);
    if (a.stage == 0) hipLaunchKernelGGL((k_ensemble<real, true>), g, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_ensemble<real, false>), g, dim3(256), 0, st, a);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_standardize(const real* y, const real* var, real* xt, int nchan, int max_len,
                              const int* chan_len, const int64_t* chan_off, hipStream_t st)
{
    hipLaunchKernelGGL((k_standardize<real>), dim3(blocks_for(max_len, 256), nchan), dim3(256), 0, st,
                       y, var, xt, chan_len, chan_off);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_channels(bool in, void* const* ptr, int nchan, int rows, int64_t max_len,
                           const int* chan_len, const int64_t* off, real* own, hipStream_t st)
{
    const unsigned bx = std::min(capped_blocks((int64_t)rows * max_len, 256), 4096u);
    for (int c = 0; c < nchan; c += kPtrBatch) {
        const int nc = std::min(kPtrBatch, nchan - c);
        PtrBatch b{};
        for (int q = 0; q < nc; ++q) b.p[q] = ptr[c + q];
        const dim3 g(bx, nc);
        if (in) hipLaunchKernelGGL((k_channels<real, true>), g, dim3(256), 0, st, b, c, rows, chan_len, off, own);
        else hipLaunchKernelGGL((k_channels<real, false>), g, dim3(256), 0, st, b, c, rows, chan_len, off, own);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <typename real>
hipError_t launch_copy(real* dst, const real* src, int64_t n, hipStream_t st)
{
    hipLaunchKernelGGL((k_copy<real>), dim3(capped_blocks(n, 256)), dim3(256), 0, st, dst, src, n);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_select_copy(const SeriesDev& sd, int max_len, const real* hA, const real* hB,
                              const int* parity, real* dst, hipStream_t st)
{
    const unsigned gy = (unsigned)(sd.nseries < 65535 ? sd.nseries : 65535);
    hipLaunchKernelGGL((k_select_copy<real>), dim3(blocks_for(max_len, 256), gy), dim3(256), 0, st,
                       sd, hA, hB, parity, dst);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_adj_tile(const AdjTileArgs<real>& a, hipStream_t st, bool force_loop)
{
    if (2 * (a.sd.cap - 2) != kWT) return hipErrorInvalidValue;
    if (const unsigned full = force_loop ? 0u : full_blocks(a.sd.ntiles, kThreads / kWave))
        hipLaunchKernelGGL((k_adj_tile<real, false>), dim3(full), dim3(kThreads), 0, st, a);
    else
        hipLaunchKernelGGL((k_adj_tile<real, true>), dim3(capped_blocks(a.sd.ntiles, kThreads / kWave)),
                           dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_adj_span_knot(const AdjArgs<real>& a, int solve_grid, hipStream_t st)
{
    hipLaunchKernelGGL((k_adj_span<real>), dim3(blocks_for(a.sd.ntiles, 256)), dim3(256), 0, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_adj_knot<real, Geom<real>::B, Geom<real>::H>), dim3(solve_grid),
                       dim3(kThreads), 0, st, a);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_adj_seed(const real* gimf, int M, int64_t N, int64_t stride, real* gr,
                           hipStream_t st)
{
    hipLaunchKernelGGL((k_adj_seed<real>), dim3(blocks_for(N, 256)), dim3(256), 0, st, gimf, M,
                       (int)N, stride, gr);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_adj_stage(int stage, int nchan, int I, int max_len, const int* chan_len,
                            const int64_t* chan_off, const SeriesDev& sd, const real* gr_next,
                            const real* mu, const real* E, const real* r_k, const real* mean_k,
                            const double* sq_k, real eps0, real* gr_k, real* gacc, real* dots,
                            real* coef, hipStream_t st)
{
    const dim3 g(blocks_for(max_len, 256), nchan);
    hipLaunchKernelGGL((k_adj_accum<real>), g, dim3(256), 0, st, I, chan_len, chan_off, sd, gr_next,
                       mu, gacc);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (stage > 0) {
        hipLaunchKernelGGL((k_adj_dot<real>), dim3(sd.nseries), dim3(1024), 0, st, I, sd, chan_off,
                           gr_next, mu, E, dots);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        hipLaunchKernelGGL((k_adj_coef<real>), dim3(nchan), dim3(kWave), 0, st, I, chan_len, dots,
                           sq_k, eps0, coef);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_adj_stage<real>), g, dim3(256), 0, st, chan_len, chan_off, gacc,
                       stage > 0 ? coef : nullptr, mean_k, r_k, gr_k);
    return hipGetLastError();
}

template <typename real>
hipError_t launch_adj_input(int nchan, const int* chan_len, const int64_t* chan_off, const real* y,
                            const real* gxt, real* gy, hipStream_t st)
{
    hipLaunchKernelGGL((k_adj_input<real>), dim3(nchan), dim3(1024), 0, st, chan_len, chan_off, y,
                       gxt, gy);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t v, int64_t n, hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_u32, dim3(capped_blocks(n, 256)), dim3(256), 0, st, p, v, n);
    return hipGetLastError();
}

hipError_t launch_knot_digest(const int* tile_series, const int* tile0, const uint64_t* mask,
                              int ntiles, uint64_t* out, int nseries, hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_u32, dim3(blocks_for(2 * (int64_t)nseries, 256)), dim3(256), 0, st,
                       (uint32_t*)out, 0u, 2 * (int64_t)nseries);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_knot_digest, dim3(blocks_for(ntiles, 256)), dim3(256), 0, st, tile_series,
                       tile0, mask, ntiles, (unsigned long long*)out);
    return hipGetLastError();
}

hipError_t launch_check_index(const int* d_x, int64_t N, int* err, hipStream_t st)
{
    hipLaunchKernelGGL(k_check_index, dim3(blocks_for(N, 256)), dim3(256), 0, st, d_x, N, err);
    return hipGetLastError();
}

#define ICM_INSTANTIATE(real)                                                                      \
    template hipError_t launch_init<real>(const SeriesDev&, const InitArgs<real>&, real*,          \
                                          const KnotsDev<real>&, const PassCtl&, hipStream_t,      \
                                          bool);                                                   \
    template hipError_t launch_sift<real>(const SiftArgs<real>&, int, hipStream_t);                \
    template hipError_t launch_knot_prefix<real>(const SeriesDev&, const KnotsDev<real>&,          \
                                                 const real*, const PassCtl&, const int*,          \
                                                 hipStream_t);                                     \
    template hipError_t launch_solve<real>(const SolveArgs<real>&, int, hipStream_t);              \
    template hipError_t launch_rilling_decide<real>(const SeriesDev&, const int*, const int*,      \
                                                    const int*, int*, int*, int*, int, int,        \
                                                    const unsigned*, unsigned*, hipStream_t);      \
    template hipError_t launch_series_var<real>(const real*, const int64_t*, int64_t, const int*,  \
                                                int, real*, real*, double*, int, hipStream_t);     \
    template hipError_t launch_noise<real>(uint64_t, int, int64_t, real*, hipStream_t);            \
    template hipError_t launch_noise_groups<real>(uint64_t, int, int, const int64_t*, const int*,  \
                                                  const int64_t*, real*, hipStream_t);             \
    template hipError_t launch_ensemble<real>(const EnsembleArgs<real>&, int, int, hipStream_t);   \
    template hipError_t launch_standardize<real>(const real*, const real*, real*, int, int,        \
                                                 const int*, const int64_t*, hipStream_t);         \
    template hipError_t launch_channels<real>(bool, void* const*, int, int, int64_t, const int*,   \
                                              const int64_t*, real*, hipStream_t);                 \
    template hipError_t launch_copy<real>(real*, const real*, int64_t, hipStream_t);               \
    template hipError_t launch_select_copy<real>(const SeriesDev&, int, const real*, const real*,  \
                                                 const int*, real*, hipStream_t);

#define ICM_INSTANTIATE_ADJ(real)                                                                  \
    template hipError_t launch_adj_tile<real>(const AdjTileArgs<real>&, hipStream_t, bool);        \
    template hipError_t launch_adj_span_knot<real>(const AdjArgs<real>&, int, hipStream_t);        \
    template hipError_t launch_adj_seed<real>(const real*, int, int64_t, int64_t, real*,           \
                                              hipStream_t);                                        \
    template hipError_t launch_adj_stage<real>(int, int, int, int, const int*, const int64_t*,     \
                                               const SeriesDev&, const real*, const real*,         \
                                               const real*, const real*, const real*,              \
                                               const double*, real, real*, real*, real*, real*,    \
                                               hipStream_t);                                       \
    template hipError_t launch_adj_input<real>(int, const int*, const int64_t*, const real*,       \
                                               const real*, real*, hipStream_t);

ICM_INSTANTIATE(float)
ICM_INSTANTIATE(double)
ICM_INSTANTIATE_ADJ(float)
ICM_INSTANTIATE_ADJ(double)

}  // namespace icm
