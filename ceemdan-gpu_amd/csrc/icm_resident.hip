// A whole sifting stage of one series in one workgroup (gfx950, wave64).
//
// The launch-per-step path of icm_kernels.hip takes three to four launches
// per pass, each a few microseconds of latency on a plan of short series.
// Here a workgroup owns a series for all passes of a stage and the steps of
// a pass are separated by workgroup barriers: the knots and the interval
// coefficients live in LDS as far as they fit, else in a scratch slice that
// the workgroup keeps in its L2.  Every arithmetic expression is the one of the
// launch-per-step kernels (icm_spline.h), on the same windows, so the two
// paths give the same bits.
//
// Layout of a series in the workgroup: a wave owns consecutive tiles of
// 256 samples, lane l the samples 64 r + l of each.  A pass is
//   samples     the stage start, or both envelopes of the previous pass at
//               the wave's own samples (and at the two samples beside them)
//               and h - mean; then the extrema of the result
//   knots       every wave ranks its knots (the waves' counts are the only
//               exchange) and writes position and value at the knot's index
//   solve       windows of 64 B knot rows, one wave each, as k_solve
//   intervals   b and d of every interval, one lane each
#include "icm_kernels.h"
#include "icm_spline.h"

#include <algorithm>
#include <cstdint>

namespace icm {
namespace {

// Entries before knot 0 and after the last knot of a type.  A window's lanes
// read the B + 2 knots around their rows without a bound test: from H + 1
// entries before knot 0 (never used by an inner row) to 17 after the last.  A
// type's entries begin at a multiple of 8 and so do the B + 2 of every lane
// (one per row and one on each side, B = 8), which are read 16 bytes at a time.
template <typename real> struct Pad {
    static constexpr int front = Geom<real>::H + 1;
    static constexpr int total = Geom<real>::H + 1 + 18;
};

// Knots and intervals of one pass: `e1` entries for the maxima, then the
// minima's; knot g of type ty is entry (ty ? e1 : 0) + front + g.  The entry
// before knot 0 repeats interval 0, for sample 0, which has no knot before it.
template <typename real>
struct KnotRows {
    real *y, *c;        // values and spline coefficients
    Coef2<real>* bd;    // b and d of the interval that starts at the knot
    uint16_t* p;        // positions (series of at most 65535 samples)
};

// Values and positions at `yp`, coefficients at `cd`.
template <typename real>
__device__ __forceinline__ KnotRows<real> knot_rows(char* yp, char* cd, int entries)
{
    // (c one entry short of the others' alignment: a lane stores it from its
    // first row, one entry after the first that it reads)
    KnotRows<real> k;
    k.y = (real*)yp;
    k.p = (uint16_t*)(k.y + entries);
    k.bd = (Coef2<real>*)cd;
    k.c = (real*)(k.bd + entries) + 7;
    return k;
}

// bytes of the first part (a multiple of 16) and of both
template <typename real>
__host__ __device__ constexpr int64_t value_bytes(int64_t entries) { return entries * ((int64_t)sizeof(real) + 2); }

template <typename real>
__host__ __device__ constexpr int64_t rows_bytes(int64_t entries)
{
    return value_bytes<real>(entries) + (3 * entries + 8) * (int64_t)sizeof(real);
}

// entries of the maxima (a multiple of 8) and of both types
template <typename real>
__host__ __device__ constexpr int64_t type_entries(int64_t n) { return (n + Pad<real>::total + 7) & ~(int64_t)7; }

// N consecutive values from a 16-byte boundary (bytes a multiple of 16, or
// the rest after those)
template <int N, typename T>
__device__ __forceinline__ void load_wide(const T* p, T (&v)[N])
{
    typedef T Vec __attribute__((ext_vector_type(16 / sizeof(T)), aligned(16)));
    constexpr int E = 16 / sizeof(T);
#pragma unroll
    for (int i = 0; i + E <= N; i += E) {
        const Vec q = *(const Vec*)(p + i);
#pragma unroll
        for (int e = 0; e < E; ++e) v[i + e] = q[e];
    }
#pragma unroll
    for (int i = N / E * E; i < N; i += 2) {
        typedef T Two __attribute__((ext_vector_type(2), aligned(2 * sizeof(T))));
        const Two q = *(const Two*)(p + i);
        v[i] = q[0];
        v[i + 1] = q[1];
    }
}

// x[q] of the lane and row that hold window row r (wave-uniform result)
template <typename real, int B>
__device__ __forceinline__ real window_row(const real (&x)[B], int r)
{
    // every row of the lane is read first: selecting among x[q] directly
    // became an indexed load, and x an array in scratch memory
    real v = lane_value(x[0], r / B);
#pragma unroll
    for (int q = 1; q < B; ++q) {
        const real u = lane_value(x[q], r / B);
        v = (r % B == q) ? u : v;
    }
    return v;
}

// Record of pass j with its pointers as ones to global memory (pointers read
// from memory are generic, and generic accesses wait for LDS as well).
template <typename T>
using Global = __attribute__((address_space(1))) T*;
struct PassRecord {
    Global<uint64_t> mask;
    Global<int> left, right, cnt, pre, n, fixf, winlist;
    unsigned* wincount;
};
__device__ __forceinline__ PassRecord record(const StageRec* rec, int j)
{
    const StageRec& r = rec[j];
    return PassRecord{(Global<uint64_t>)r.mask, (Global<int>)r.left, (Global<int>)r.right,
                      (Global<int>)r.cnt, (Global<int>)r.pre, (Global<int>)r.n, (Global<int>)r.fixf,
                      (Global<int>)r.winlist, r.wincount};
}

// Solves window w of the n knots of type ty (entries from e0 = knot 0) and
// writes c of the rows it keeps; the window that keeps an end knot stores the
// end values after the endpoint fix in fix[0..1].  Not-a-knot ends change
// rows 1 and n - 2 only: their entries are wave-uniform, selected per row.
// A short series has one window per type, so a pass waits for the serial
// chain and the issue slots of one wave here (half of it): 7.7 -> 5.2 thousand
// cycles in FP64, 5.3 -> 3.1 in FP32, with the entries in 16-byte reads
// (eight lanes met in a bank before), both ends at once in even and odd lanes,
// no branch among the rows, pivots without operand scaling and the levels of
// partition_pcr that change nothing left out.
template <typename real, bool NAK>
__device__ __forceinline__ void solve_window(const KnotRows<real>& k, int e0, int ty, int n, int w,
                                             int lane, real* fix, Global<int> fixf)
{
    constexpr int B = Geom<real>::B, H = Geom<real>::H, W = kWave * B, K = W - 2 * H;
    const int g0 = w * K - H, lo = g0 - 1;
    const int rb = lane * B;
    // knots 0, 1, 2 (even lanes) or n-1, n-2, n-3 (odd lanes): the two ends
    // are mirror images with the same arithmetic, bit for bit
    const bool odd = lane & 1;
    const int i0 = e0 + (odd ? n - 1 : 0), i1 = e0 + (odd ? n - 2 : 1), i2 = e0 + (odd ? max(n - 3, 0) : min(2, n - 1));
    const int he = (int)k.p[i1] - (int)k.p[i0], hn = (int)k.p[i2] - (int)k.p[i1];
    const real y0 = k.y[i0], y1 = k.y[i1], y2 = k.y[i2];
    uint16_t px[B + 2];
    real py[B + 2];
    {
        const int at = e0 + lo + min(rb, (n - lo + 7) & ~7);
        load_wide(k.p + at, px);
        load_wide(k.y + at, py);
    }
    int hx[B + 1];
    real sl[B + 1];
#pragma unroll
    for (int j = 0; j <= B; ++j) {
        hx[j] = (int)px[j + 1] - (int)px[j];
        sl[j] = sdiv<real>(py[j + 1] - py[j], (real)hx[j]);
    }
    // endpoint fix from the line through the two knots next to the end
    // (setBoundaryMax/Min, cudaICEEMDAN.cu:209-291), and the slopes of the
    // first and last interval with it
    {
        const real t = y1 - (y2 - y1) / (real)hn * (real)he;
        const bool above = t > y0, below = t < y0;
        const bool take = n >= 6 && (ty == 0 ? above : below);
        const real v = take ? t : y0;
        const real se = sdiv<real>(y1 - v, (real)he);
        const real sa = lane_value(se, 0), sz = lane_value(se, 1);
        constexpr int j0 = (H + 1) % B;
        sl[j0] = lo + rb + j0 == 0 ? sa : sl[j0];
        const int jz = n - 2 - lo - rb;
#pragma unroll
        for (int j = 0; j <= B; ++j) sl[j] = j == jz ? sz : sl[j];
        // stored by the window that keeps the end
        const int ge = odd ? n - 1 : 0;
        if (lane < 2 && ge >= w * K && ge < w * K + K) {
            fix[lane] = v;
            if (fixf) fixf[lane] = take ? 1 : 0;
        }
    }
    // rows of not-a-knot ends: (dl, d, du) of row 1 and of row n - 2
    int gn1 = -1, gn2 = -1;
    real d1 = (real)1, u1 = (real)0, l2 = (real)0, d2 = (real)1;
    if (NAK) {
        const int ae = abs(he), an = abs(hn);
        const real dd = (real)(3 * ae + 2 * an) + (real)ae * (real)ae / (real)an;
        const real oo = (real)an - (real)ae * (real)ae / (real)an;
        gn1 = 1;
        gn2 = n - 2;
        d1 = lane_value(dd, 0);
        u1 = lane_value(oo, 0);
        d2 = lane_value(dd, 1);
        l2 = lane_value(oo, 1);
    }
    real xs[B];
    partition_pcr<real, B, !NAK>(
        lane,
        [&](int q, real& dl, real& d, real& du, real& f) {
            const int g = g0 + rb + q;
            spline_row<real, false>(n, g, hx[q], hx[q + 1], sl[q], sl[q + 1], dl, d, du, f);
            if (NAK) {
                // n >= 4, so rows 1 and n - 2 are different rows
                d = g == gn1 ? d1 : g == gn2 ? d2 : d;
                du = g == gn1 ? u1 : g == gn2 ? (real)0 : du;
                dl = g == gn1 ? (real)0 : g == gn2 ? l2 : dl;
            }
        },
        xs);
    // whole lanes keep their rows; a lane's rows past the last knot land in
    // its tail padding
    if (lane >= H / B && lane < kWave - H / B && g0 + rb < n) {
        typedef real Vec __attribute__((ext_vector_type(16 / sizeof(real)), aligned(16)));
        constexpr int E = 16 / sizeof(real);
#pragma unroll
        for (int q = 0; q < B; q += E) {
            Vec v;
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = xs[q + e];
            *(Vec*)(k.c + e0 + g0 + rb + q) = v;
        }
    }
    if (NAK) {
        // the window that keeps an end knot recovers it from its own rows
        const int r0 = -g0, r1 = n - 1 - g0;
        if (r0 >= H && r0 < H + K) {
            const real c1 = window_row<real, B>(xs, r0 + 1), c2 = window_row<real, B>(xs, r0 + 2);
            if (lane == 0) k.c[e0] = nak_end<real>(c1, c2, he, hn);
        }
        if (r1 >= H && r1 < H + K) {
            const real c1 = window_row<real, B>(xs, r1 - 1), c2 = window_row<real, B>(xs, r1 - 2);
            if (lane == 1) k.c[e0 + n - 1] = nak_end<real>(c1, c2, -he, -hn);
        }
    }
}

// b and d of the intervals of both types (spline_coefficients,
// cudaICEEMDAN.cu:394-398); interval 0 also into the entry before it, with
// the fixed value of its knot
template <typename real, int NT>
__device__ __forceinline__ void intervals(const KnotRows<real>& k, int e1, const int (&n)[2],
                                          const real (*fix)[2])
{
    for (int q = threadIdx.x; q < n[0] + n[1] - 2; q += NT) {
        const bool ty = q >= n[0] - 1;
        const int g = ty ? q - (n[0] - 1) : q;
        const int e = (ty ? e1 : 0) + Pad<real>::front + g;
        real a0 = k.y[e], a1 = k.y[e + 1];
        const real c0 = k.c[e], c1 = k.c[e + 1];
        const int p0 = k.p[e], p1 = k.p[e + 1];
        const real f0 = fix[ty][0], f1 = fix[ty][1];
        a0 = g == 0 ? f0 : a0;
        a1 = g == (ty ? n[1] : n[0]) - 2 ? f1 : a1;
        Coef2<real> bd;
        interval_bd<real>((real)(p1 - p0), a0, a1, c0, c1, bd.b, bd.d);
        k.bd[e] = bd;
        if (g == 0) {
            k.y[e] = a0;
            k.y[e - 1] = a0;
            k.c[e - 1] = c0;
            k.bd[e - 1] = bd;
            k.p[e - 1] = (uint16_t)p0;
        }
    }
}

// envelope at sample p, e the entry of its interval
template <typename real>
__device__ __forceinline__ real envelope(const KnotRows<real>& k, int p, int e)
{
    const Coef2<real> bd = k.bd[e];
    const Coef<real> q{k.y[e], bd.b, k.c[e], bd.d};
    return horner(q, (real)(p - (int)k.p[e]));
}

// x_i of the stage start at four samples and one beside them, one straight
// line of loads per start mode (init_load of icm_kernels.hip)
template <typename real>
struct Start {
    using P = typename Promote<real>::type;
    const real *src, *E;
    P scl0;
    real sclk, eps0;
    int mode;
    template <int NS>
    __device__ __forceinline__ void at(const int (&p)[NS], real (&v)[NS]) const
    {
        if (mode == INIT_COPY || mode == INIT_KNOTS) {
#pragma unroll
            for (int i = 0; i < NS; ++i) v[i] = src[p[i]];
            return;
        }
        real e[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            v[i] = src[p[i]];
            e[i] = E[p[i]];
        }
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            if (mode == INIT_RESID) v[i] = v[i] - e[i];
            else if (mode == INIT_STAGE0) v[i] = (real)((P)v[i] + (P)(eps0 * e[i]) * scl0);
            else v[i] = v[i] + (eps0 * e[i]) * sclk;
        }
    }
};

enum StageKind : int { STAGE_FIXED = 0, STAGE_RECORD = 1, STAGE_RILLING = 2 };

// inclusive sum over the lanes of each 16-lane row
__device__ __forceinline__ int row_scan(int v)
{
    v += dpp_row_i<0x111, 0xF>(v, 0);
    v += dpp_row_i<0x112, 0xF>(v, 0);
    v += dpp_row_i<0x114, 0xF>(v, 0);
    v += dpp_row_i<0x118, 0xF>(v, 0);
    return v;
}

// HOLD: every wave owns at most one tile, whose samples stay in registers
// from pass to pass; else a wave goes through its tiles (at most 8: their row
// masks fill the 64 lanes of one register pair) and reads its own samples
// back from the series' buffer.
template <typename real, int NWV, bool HOLD, int KIND>
__global__ __launch_bounds__(NWV* kWave) __attribute__((amdgpu_waves_per_eu(4)))
void k_stage(StageArgs<real> a)
{
    using P = typename Promote<real>::type;
    constexpr int B = Geom<real>::B, H = Geom<real>::H, K = kWave * B - 2 * H;
    constexpr int NT = NWV * kWave, F = Pad<real>::front;
    constexpr bool RILL = KIND == STAGE_RILLING, REC = KIND == STAGE_RECORD;
    extern __shared__ __align__(16) char smem[];
    __shared__ int s_tot[NWV];
    __shared__ real s_edge[2][NWV][2];
    __shared__ real s_fix[2][2];
    __shared__ int s_sx[NWV][2];
    const int lane = threadIdx.x & 63, wv = wave_index();
    char* const scratch = HOLD ? nullptr : a.scratch + (int64_t)blockIdx.x * a.slot_bytes;

    for (int s = blockIdx.x; s < a.nseries; s += gridDim.x) {
        const bool uni = a.sd.len == nullptr;
        const int N = uni ? a.uniform_len : a.sd.len[s];
        const int64_t off = uni ? (int64_t)s * N : a.sd.off[s];
        const int ntl = (N + kWT - 1) / kWT;
        // tiles of this wave: the first waves have one more where they do not
        // divide evenly (waves go to the SIMDs in turn, so these share alike;
        // with ceil(tiles / waves) for all but the last, a sparse pass of 10007
        // FP32 samples took 25.4 thousand cycles instead of 22.1, of 30504 60.1
        // instead of 56.9)
        const int rest = ntl % NWV, t_first = wv * (ntl / NWV) + min(wv, rest);
        const int nt = ntl / NWV + (wv < rest ? 1 : 0);
        const int start = t_first * kWT, end = min(start + nt * kWT, N);
        // sample buffers: RILLING alternates hA and hB (a series that stops
        // at pass j exports the input of pass j); FIXED keeps one
        real* const buf0 = a.hA + off;
        real* const buf1 = RILL ? a.hB + off : buf0;

        real hv[kWR];           // HOLD: the wave's samples
        uint64_t mk = 0;        // lane 32 ty + row: the wave's knot row masks
        int base[2] = {0, 0}, n[2] = {0, 0}, tot[2] = {0, 0};
        int e1 = 0, entries = 0;
        bool in_lds = true;
        int stop = 0;

        // row masks of the strict extrema of tile tl (nx: a vector whose lane
        // 0 is the sample after the tile); cg, cl: the comparisons of the
        // sample before the row with the row's first
        uint64_t cg = 0, cl = 0;
        auto extrema = [&](int tl, const real (&v)[kWR], real nx) {
            uint64_t gt[kWR], lt[kWR];
#pragma unroll
            for (int r = 0; r < kWR; ++r) {
                const real rgt = row_next(v[r], r < kWR - 1 ? v[r < kWR - 1 ? r + 1 : r] : nx);
                gt[r] = wave_ballot(v[r] > rgt);
                lt[r] = wave_ballot(v[r] < rgt);
            }
            const int t0 = start + tl * kWT;
            const bool ends = t0 == 0 || t0 + kWT >= N;
#pragma unroll
            for (int r = 0; r < kWR; ++r) {
                // a comparison of neighbours p, p + 1 serves both samples
                uint64_t mx = gt[r] & ((lt[r] << 1) | cl), mn = lt[r] & ((gt[r] << 1) | cg);
                cg = gt[r] >> 63;
                cl = lt[r] >> 63;
                if (ends) {
                    const int p0 = t0 + r * kWave, left = N - p0;   // samples from the row's first
                    uint64_t e = p0 == 0 ? 1ull : 0ull;
                    if (left >= 1 && left <= 64) e |= 1ull << (left - 1);
                    const uint64_t valid = left >= 64 ? ~0ull : left <= 0 ? 0ull : (1ull << left) - 1;
                    mx = valid & (e | mx);
                    mn = valid & (e | mn);
                }
                tot[0] += __popcll(mx);
                tot[1] += __popcll(mn);
                set_lane(mk, mx, tl * kWR + r);
                set_lane(mk, mn, 32 + tl * kWR + r);
            }
        };
        auto first_row = [&](real el, real v0) {
            cg = wave_ballot(el > v0) & 1ull;
            cl = wave_ballot(el < v0) & 1ull;
        };
        auto store = [&](real* dst, int tl, const real (&v)[kWR]) {
            const int p0 = start + tl * kWT + lane;
            if (start + tl * kWT + kWT <= N) {
#pragma unroll
                for (int r = 0; r < kWR; ++r) dst[p0 + r * kWave] = v[r];
            } else {
#pragma unroll
                for (int r = 0; r < kWR; ++r)
                    if (p0 + r * kWave < N) dst[p0 + r * kWave] = v[r];
            }
        };
        auto fetch = [&](const real* src, int tl, real (&v)[kWR]) {
            const int p0 = start + tl * kWT + lane;
#pragma unroll
            for (int r = 0; r < kWR; ++r) v[r] = src[min(p0 + r * kWave, N - 1)];
        };
        // the wave's samples at the edges, for its neighbours
        auto publish = [&](int par, real first, real last) {
            if (lane == 0) s_edge[par][wv][0] = first;
            if (lane == 63) s_edge[par][wv][1] = last;
        };

        // ---- stage start
        {
            Start<real> in{};
            in.mode = a.ia.mode;
            in.eps0 = a.ia.eps0;
            if (in.mode == INIT_STAGE0 || in.mode == INIT_STAGEK) {
                const int c = a.sd.chan[s];
                in.src = a.ia.chan_sig + a.ia.chan_off[c];
                in.E = a.ia.E + a.sd.eoff[s];
                if (in.mode == INIT_STAGE0) in.scl0 = (P)a.ia.scale[a.sd.nidx[s]];
                else in.sclk = (real)a.ia.scale[c];
            } else {
                in.src = a.ia.src + off;
                if (in.mode == INIT_RESID) in.E = a.ia.E + off;
            }
            auto load = [&](int tl, real (&v)[kWR]) {
                const int p0 = start + tl * kWT + lane;
                int p[kWR];
#pragma unroll
                for (int r = 0; r < kWR; ++r) p[r] = min(p0 + r * kWave, N - 1);
                in.at(p, v);
                if (in.mode == INIT_RESID) store(a.ia.resid + off, tl, v);
                if (RILL || !HOLD) store(buf0, tl, v);
            };
            if (nt > 0) {
                int pe[1] = {lane == 0 ? max(start - 1, 0) : min(end, N - 1)};
                real ve[1];
                in.at(pe, ve);
                const real el = lane_value(ve[0], 0), er = lane_value(ve[0], 1);
                if constexpr (HOLD) {
                    load(0, hv);
                    first_row(el, hv[0]);
                    extrema(0, hv, er);
                    publish(0, hv[0], hv[kWR - 1]);
                } else {
                    real prev[kWR], v[kWR];
                    load(0, v);
                    first_row(el, v[0]);
                    const real first = v[0];
                    for (int tl = 1; tl <= nt; ++tl) {
#pragma unroll
                        for (int r = 0; r < kWR; ++r) prev[r] = v[r];
                        if (tl < nt) load(tl, v);
                        extrema(tl - 1, prev, tl < nt ? v[0] : er);
                    }
                    publish(0, first, prev[kWR - 1]);
                }
            }
        }

        int sxc = 0;
        bool sxm = false;
        for (int j = 0;; ++j) {
            // knots of the input of pass j are flagged
            if (lane == 0) {
                s_tot[wv] = tot[0] | (tot[1] << 16);
                if (RILL) {
                    s_sx[wv][0] = sxc;
                    s_sx[wv][1] = sxm;
                }
            }
            __syncthreads();
            if (RILL && j > 0) {
                // stop rule of pass j - 1 (siftingCriterion, cudaICEEMDAN.cu:494-525)
                const int c = lane_value_i(row_scan(s_sx[lane & (NWV - 1)][0]), NWV - 1);
                const bool m = wave_ballot(s_sx[lane & (NWV - 1)][1] != 0) != 0ull;
                const real frac = (real)(long long)c * (real)(1.0 / (double)N);
                if (!((frac > (real)0.05) || (m && n[0] + n[1] > 6))) {
                    stop = j - 1;
                    break;
                }
            }
            {
                const int v = row_scan(s_tot[lane & (NWV - 1)]);
                const int all = lane_value_i(v, NWV - 1), own = lane_value_i(v, wv);
                n[0] = all & 0xFFFF;
                n[1] = (int)((unsigned)all >> 16);
                base[0] = (own & 0xFFFF) - tot[0];
                base[1] = (int)((unsigned)own >> 16) - tot[1];
            }
            if (a.nk_out && j == 0 && threadIdx.x < 2) a.nk_out[2 * s + threadIdx.x] = threadIdx.x ? n[1] : n[0];
            if (RILL && j == a.passes - 1) {
                stop = j;      // the cap: the input of this pass is exported
                break;
            }
            const bool use_mean = n[0] > 3 && n[1] > 3;
            e1 = (int)type_entries<real>(n[0]);
            entries = e1 + (int)type_entries<real>(n[1]);
            in_lds = HOLD || rows_bytes<real>(entries) <= a.lds_bytes;
            const bool last = !RILL && j == a.passes - 1;
            const real* const hin = j & 1 ? buf1 : buf0;                        // input of pass j
            real* const hout = last ? a.out + off : j & 1 ? buf0 : buf1;
            const bool done = last && !a.need_out;     // records only

            // the rest of the pass on rows in LDS or in the scratch slice
            auto pass = [&](const KnotRows<real> kr) {
                // ---- knots by index
                {
                    int rb[2] = {base[0] + F, base[1] + F + e1};
                    real nx[kWR];
                    if constexpr (!HOLD) {
                        if (nt > 0) fetch(hin, 0, nx);
                    }
                    for (int tl = 0; tl < nt; ++tl) {
                        const int t0 = start + tl * kWT;
                        if constexpr (!HOLD) {
                            // the next tile is requested before this one is used
#pragma unroll
                            for (int r = 0; r < kWR; ++r) hv[r] = nx[r];
                            if (tl + 1 < nt) fetch(hin, tl + 1, nx);
                        }
                        const int before[2] = {rb[0], rb[1]};
#pragma unroll
                        for (int r = 0; r < kWR; ++r) {
#pragma unroll
                            for (int ty = 0; ty < 2; ++ty) {
                                const uint64_t m = lane_value(mk, 32 * ty + tl * kWR + r);
                                const int e = rank_below(m, rb[ty]);
                                if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                                    kr.p[e] = (uint16_t)(t0 + r * kWave + lane);
                                    kr.y[e] = hv[r];
                                }
                                rb[ty] += __popcll(m);
                            }
                        }
                        if (REC && lane < 2) {
                            const int gt = (uni ? s * ntl : a.sd.tile0[s]) + t_first + tl;
                            const PassRecord R = record(a.rec, j);
                            R.pre[2 * gt + lane] = (lane ? before[1] - e1 : before[0]) - F;
                            R.cnt[2 * gt + lane] = lane ? rb[1] - before[1] : rb[0] - before[0];
                        }
                    }
                    if (REC) {
                        // the wave's row masks, [tile][type][row]
                        const int row = lane & 31;
                        const int gt = (uni ? s * ntl : a.sd.tile0[s]) + t_first + row / kWR;
                        if (row < nt * kWR)
                            record(a.rec, j).mask[8 * (int64_t)gt + kWR * (lane >> 5) + row % kWR] = mk;
                    }
                }
                __syncthreads();
                // ---- windows of the spline system
                const int wmx = (n[0] + K - 1) / K, wmn = (n[1] + K - 1) / K;
                if (REC) {
                    // by the last waves: the first ones have the windows (11 stages
                    // of 3200 series of 16384 FP64 samples: 32.6 ms unrecorded,
                    // recorded by the first waves 39.8, by the last 38.0)
                    const PassRecord R = record(a.rec, j);
                    const int gt0 = uni ? s * ntl : a.sd.tile0[s];
                    if (threadIdx.x < 2) R.n[2 * s + threadIdx.x] = threadIdx.x ? n[1] : n[0];
                    for (int q = NT - 1 - threadIdx.x; q < 2 * ntl; q += NT) {
                        const int t = q >> 1, ty = q & 1, at = 2 * (gt0 + t) + ty;
                        const int pre = R.pre[at], nx = pre + R.cnt[at];
                        const int e0 = (ty ? e1 : 0) + F;
                        R.left[at] = pre > 0 ? (int)kr.p[e0 + pre - 1] : -1;
                        R.right[at] = nx < (ty ? n[1] : n[0]) ? (int)kr.p[e0 + nx] : -1;
                    }
                    if (wv == NWV - 1) {
                        unsigned wb = 0;
                        if (lane == 0) wb = atomicAdd(R.wincount, (unsigned)(wmx + wmn));
                        wb = (unsigned)__builtin_amdgcn_readfirstlane((int)wb);
                        for (int w = lane; w < wmx + wmn; w += kWave) {
                            const int ty = w >= wmx, wi = ty ? w - wmx : w;
                            const int g = max(wi * K - H - 1, 0);
                            const Global<int> item = R.winlist + kWinItem * (int64_t)(wb + w);
                            item[0] = s;
                            item[1] = (wi << 1) | ty;
                            item[2] = (int)kr.p[(ty ? e1 : 0) + F + g] / kWT;   // tile of its first knot
                        }
                    }
                }
                for (int w = wv; w < wmx + wmn; w += NWV) {
                    const int ty = w >= wmx, wi = ty ? w - wmx : w;
                    const int nty = ty ? n[1] : n[0];
                    const Global<int> fixf = REC ? record(a.rec, j).fixf + 4 * s + 2 * ty : nullptr;
                    if (a.nak && nty >= 4)
                        solve_window<real, true>(kr, (ty ? e1 : 0) + F, ty, nty, wi, lane, s_fix[ty], fixf);
                    else
                        solve_window<real, false>(kr, (ty ? e1 : 0) + F, ty, nty, wi, lane, s_fix[ty], fixf);
                }
                __syncthreads();
                if (done) return;
                intervals<real, NT>(kr, e1, n, s_fix);
                __syncthreads();
                // ---- envelopes, mean, h - m (interpolate :403-439,
                // averageUppperLower :441-454, updateRealizations :527-544)
                sxc = 0;
                sxm = false;
                if (nt == 0) return;
                const uint64_t omk = mk;    // knots of the input
                int rb[2] = {base[0] + F - 1, base[1] + e1 + F - 1};
                auto sift = [&](int tl, real (&v)[kWR]) {
                    if (RILL || use_mean) {
                        const int p0 = start + tl * kWT + lane;
                        int e[2][kWR];
#pragma unroll
                        for (int r = 0; r < kWR; ++r) {
#pragma unroll
                            for (int ty = 0; ty < 2; ++ty) {
                                const uint64_t m = lane_value(omk, 32 * ty + tl * kWR + r);
                                e[ty][r] = rank_below(m, rb[ty]);
                                rb[ty] += __popcll(m);
                            }
                        }
#pragma unroll
                        for (int r = 0; r < kWR; ++r) {
                            const int p = p0 + r * kWave;
                            const real U = envelope(kr, p, e[0][r]), L = envelope(kr, p, e[1][r]);
                            if (use_mean) v[r] = v[r] - (U + L) / (real)2;
                            if (RILL) {
                                const real sx = fabs((U + L) / (U - L));
                                sxc += __popcll(wave_ballot(p < N && sx > (real)0.05));
                                sxm |= wave_ballot(p < N && sx > (real)0.5) != 0ull;
                            }
                        }
                    }
                    if (last || RILL || !HOLD) store(hout, tl, v);
                };
                real el = (real)0, er = (real)0;
                if (!last) {
                    // the samples beside the wave's: lane 0 the one before,
                    // the others the one after; a knot lies on the interval
                    // to its left
                    const int p = lane == 0 ? start - 1 : end;
                    const int ew = lane == 0 ? max(wv - 1, 0) : min(wv + 1, NWV - 1);
                    const int b0 = base[0] + (lane == 0 ? 0 : tot[0]), b1 = base[1] + (lane == 0 ? 0 : tot[1]);
                    real v = s_edge[j & 1][ew][lane == 0 ? 1 : 0];
                    int i0 = b0 + F - 1, i1 = b1 + F - 1 + e1;
                    const int q0 = kr.p[i0], q1 = kr.p[i1];
                    i0 = q0 == p && b0 > 0 ? i0 - 1 : i0;
                    i1 = q1 == p && b1 > 0 ? i1 - 1 : i1;
                    const real U = envelope(kr, p, i0), L = envelope(kr, p, i1);
                    v = use_mean ? v - (U + L) / (real)2 : v;
                    el = lane_value(v, 0);
                    er = lane_value(v, 1);
                    mk = 0;
                    tot[0] = tot[1] = 0;
                }
                if constexpr (HOLD) {
                    sift(0, hv);
                    if (!last) {
                        first_row(el, hv[0]);
                        extrema(0, hv, er);
                        publish((j + 1) & 1, hv[0], hv[kWR - 1]);
                    }
                } else {
                    real prev[kWR], v[kWR], nx[kWR];
                    fetch(hin, 0, v);
                    if (nt > 1) fetch(hin, 1, nx);
                    sift(0, v);
                    if (!last) first_row(el, v[0]);
                    const real first = v[0];
                    for (int tl = 1; tl <= nt; ++tl) {
#pragma unroll
                        for (int r = 0; r < kWR; ++r) {
                            prev[r] = v[r];
                            v[r] = nx[r];
                        }
                        // the tile after next is requested before this one
                        if (tl + 1 < nt) fetch(hin, tl + 1, nx);
                        if (tl < nt) sift(tl, v);
                        if (!last) extrema(tl - 1, prev, tl < nt ? v[0] : er);
                    }
                    if (!last) publish((j + 1) & 1, first, prev[kWR - 1]);
                }
            };
            // rows too long for LDS keep values and positions there and the
            // coefficients in scratch where that fits (dense pass of 30504 FP32
            // samples 130.7 -> 112.0 thousand cycles, of 16384 FP64 111 -> 85.5)
            char* const behind = smem + value_bytes<real>(entries);
            if (HOLD || in_lds) pass(knot_rows<real>(smem, behind, entries));
            else if (value_bytes<real>(entries) <= a.lds_bytes) pass(knot_rows<real>(smem, scratch, entries));
            else pass(knot_rows<real>(scratch, scratch + value_bytes<real>(entries), entries));
            if (last) break;
        }
        if (RILL && threadIdx.x == 0) {
            a.stop_pass[s] = stop;
            a.subs[s] = stop;
        }
        __syncthreads();   // the next series reuses the shared arrays
    }
}

template <typename real, int NWV, bool HOLD>
void launch_one(const StageArgs<real>& a, unsigned grid, size_t lds, hipStream_t st)
{
    const dim3 g(grid), b(NWV * kWave);
    if (a.rilling) hipLaunchKernelGGL((k_stage<real, NWV, HOLD, STAGE_RILLING>), g, b, lds, st, a);
    else if (a.rec) hipLaunchKernelGGL((k_stage<real, NWV, HOLD, STAGE_RECORD>), g, b, lds, st, a);
    else hipLaunchKernelGGL((k_stage<real, NWV, HOLD, STAGE_FIXED>), g, b, lds, st, a);
}

}  // namespace

// Which phases take the stage kernel, and its workgroup.  Measured per pass
// (us, the CEEMDAN stages of a replayed decomposition of one EEG-like channel
// with their sums) against the tuned launch-per-step path:
//   series x samples    FP32 steps / stage     FP64 steps / stage
//     50 x   1000           27.6 / 5.2             31.5 / 6.8
//   4000 x   1000          132.1 / 50.8           152.5 / 67.9
//     50 x   4000           28.5 / 6.7             34.3 / 9.0
//   4000 x   4000          179.9 / 102.1          235.0 / 148.3
//   4000 x   8000          245.8 / 183.5          347.6 / 289.0
//   3000 x  16000          295.9 / 243.5          433.8 / 363.2
//      4 x  24000           34.0 / 23.4            39.5 / 34.7
//     50 x  24000           39.4 / 24.3            47.2 / 37.4
//    500 x  24000           89.4 / 56.4           126.4 / 87.9
//   3000 x  24000          411.2 / 335.0          605.2 / 508.0
//      4 x  32000           34.9 / 30.6            42.0 / 47.7
//     50 x  32000           41.8 / 32.0            49.1 / 51.8
//    100 x  32000           46.0 / 35.8            59.9 / 54.3
//    250 x  32000           70.7 / 39.6            95.3 / 68.7
//    500 x  32000          108.4 / 77.2           155.1 / 134.9
//    800 x  32000          153.4 / 145.1          232.0 / 253.1 (an earlier state)
//   3000 x  32000          527.5 / 459.9          783.6 / 806.8 (an earlier state)
// A workgroup sifts one series at a time and one fits a CU from about 2000
// samples on, so its time grows with series / 256 and is flat below 256, while
// the launch-per-step path spreads any one pass over the chip: FP64 series of
// more than 96 tiles lose here beyond three workgroups per CU, and long ones
// where they or their rows are few (few_long_series in icm_plan.hip).
// Waves per workgroup: one tile each as far as 16 waves go (the shortest
// pass); FP32 series of up to 16 tiles in plans of more series than CUs take
// 8 waves, so that two workgroups share a CU (500 x 4000: 11.8 against 13.4).
StageGeom stage_geometry(int real_size, int64_t max_len, int64_t nseries)
{
    StageGeom g{};
    const bool f64 = real_size == 8;
    const int64_t ntl = (max_len + kWT - 1) / kWT;
    const int64_t most_series = ntl > 128 ? 0 : f64 && ntl > 96 ? 768 : INT64_MAX;
    if (nseries > most_series) return g;
    g.nwv = ntl <= 4 ? 4 : ntl <= 8 || (!f64 && ntl <= 16 && nseries > 256) ? 8 : 16;
    g.hold = ntl <= g.nwv;
    // knot rows of the densest pass (at most N + 4 knots of both types)
    const int64_t entries = max_len + 4 + 2 * (f64 ? type_entries<double>(0) : type_entries<float>(0)) + 16;
    const size_t worst = (size_t)(f64 ? rows_bytes<double>(entries) : rows_bytes<float>(entries));
    const size_t most = 160 * 1024 - 2048;     // static arrays aside
    g.lds = std::min(worst, most);
    g.slot = worst <= most ? 0 : (worst + 255) / 256 * 256;
    // with scratch one workgroup per CU; else one per series, up to a grid of
    // at most 2^30 work-items (a workgroup goes on to the next series)
    g.grid = std::min<int64_t>(nseries, g.slot ? 256 : 1 << 20);
    g.ok = true;
    return g;
}

template <typename real>
hipError_t launch_stage(const StageArgs<real>& args, const StageGeom& g, hipStream_t st)
{
    StageArgs<real> a = args;
    a.lds_bytes = (int)g.lds;
    a.slot_bytes = (int64_t)g.slot;
    const unsigned grid = (unsigned)g.grid;
    if (g.nwv == 4 && g.hold) launch_one<real, 4, true>(a, grid, g.lds, st);
    else if (g.nwv == 8 && g.hold) launch_one<real, 8, true>(a, grid, g.lds, st);
    else if (g.hold) launch_one<real, 16, true>(a, grid, g.lds, st);
    else if (g.nwv == 16) launch_one<real, 16, false>(a, grid, g.lds, st);
    else if constexpr (sizeof(real) == 4) launch_one<real, 8, false>(a, grid, g.lds, st);   // FP32 only
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

template hipError_t launch_stage<float>(const StageArgs<float>&, const StageGeom&, hipStream_t);
template hipError_t launch_stage<double>(const StageArgs<double>&, const StageGeom&, hipStream_t);

}  // namespace icm
