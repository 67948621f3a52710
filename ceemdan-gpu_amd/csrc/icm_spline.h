// Arithmetic shared by the sift kernels: spline rows, the windowed partition +
// PCR solve, interval coefficients and envelope evaluation (gfx950, wave64).
// Both forward paths (one launch per step of a pass, or one workgroup per
// series for a whole stage) build on these functions, so they round alike.
#pragma once
#include "icm_device.h"

#include <type_traits>

namespace icm {

// promotion type used where the reference mixes float data with double
// literals (cudaICEEMDAN.cu:50, :64, :76); identity for double
template <typename real> struct Promote { using type = double; };

constexpr int kWT = 256;               // samples per tile
constexpr int kWR = kWT / kWave;       // 64-sample chunks per tile

// orders this wave's LDS and memory accesses before and after it
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// base + the number of set bits of `mask` below this lane (two mbcnt steps;
// running bases instead of a per-row prefix array keep eight scalar
// registers free, which the sift loop would otherwise spill)
__device__ __forceinline__ int rank_below(uint64_t mask, int base)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, (uint32_t)base));
}

// ------------------------------------------------------- interval coefficients

// Interval coefficients S(t) = a + (b + (c + d t) t) t, t = p - pos.
template <typename real>
struct alignas(2 * sizeof(real)) Coef {
    real a, b, c, d;
};

template <typename real>
struct alignas(2 * sizeof(real)) Coef2 {
    real b, d;
};

// Horner steps as fused multiply-adds (single rounding each), the way nvcc
// contracts the reference's a + (b + (c + d t) t) t (cudaICEEMDAN.cu:436);
// the oracle evaluates the same fma chain.
template <typename real>
__device__ __forceinline__ real horner(const Coef<real>& q, real t)
{
    return fma(fma(fma(q.d, t, q.c), t, q.b), t, q.a);
}

// b and d of an interval of length hk from the values a0, a1 and the
// coefficients c0, c1 at its ends (spline_coefficients, cudaICEEMDAN.cu:394-398)
template <typename real>
__device__ __forceinline__ void interval_bd(real hk, real a0, real a1, real c0, real c1, real& b,
                                            real& d)
{
    if (std::is_same<real, double>::value) {
        // the reference's expressions, correctly rounded divisions: FP64
        // equals the oracle bit for bit
        b = (a1 - a0) / hk - hk * ((real)2 * c0 + c1) / (real)3;
        d = (c1 - c0) / ((real)3 * hk);
    } else {
        // FP32 (compared with the FP64 oracle by its error, not bit for bit):
        // the hardware reciprocal of the spacing (1 ulp) and 1/3 as a product,
        // instead of three correctly rounded divisions (~9 instructions each)
        // -- 9 % of the sift pass's time at the 64-channel FP32 job
        const real rh = (real)__builtin_amdgcn_rcpf((float)hk);
        const real third = (real)(1.0 / 3.0);
        b = (a1 - a0) * rh - hk * ((real)2 * c0 + c1) * third;
        d = (c1 - c0) * third * rh;
    }
}

// ------------------------------------------------------- windowed spline solve

template <typename real> struct Geom;
template <> struct Geom<double> { static constexpr int B = 8, H = 32; };
template <> struct Geom<float> { static constexpr int B = 8, H = 16; };

// Row g of the spline system (cudaICEEMDAN.cu:310-343) from the lengths
// hl, hr of the intervals left and right of knot g and their slopes sl, sr
// ((y_g - y_{g-1}) / hl and (y_{g+1} - y_g) / hr, each computed once per
// interval and shared by the two rows it touches); rows outside [0, n) and
// the two end rows are identity rows with a zero right-hand side.
// Not-a-knot ends (NAK, n >= 4): c_0 is eliminated from row 1 and c_{n-1}
// from row n-2 (both stay diagonally dominant); the end values follow from
// nak_end after the solve.
template <typename real, bool NAK>
__device__ __forceinline__ void spline_row(int n, long g, int hl, int hr, real sl, real sr,
                                           real& dl, real& d, real& du, real& f)
{
    // computed on every lane and selected at the end (an early return here
    // kept the four outputs in scratch memory); rows outside (0, n-1) see
    // neighbours that exist in the window's LDS but take the identity row
    const bool inner = g > 0 && g < n - 1;
    real tdl = (real)hl;
    real tdu = (real)hr;
    real td = (real)(2 * (hl + hr));
    const real tf = (real)3 * (sr - sl);
    if (NAK && n >= 4) {
        if (g == 1) {
            tdl = (real)0;
            td = (real)(3 * hl + 2 * hr) + (real)hl * (real)hl / (real)hr;
            tdu = (real)hr - (real)hl * (real)hl / (real)hr;
        }
        if (g == n - 2) {
            tdl = (real)hl - (real)hr * (real)hr / (real)hl;
            td = (real)(2 * hl + 3 * hr) + (real)hr * (real)hr / (real)hl;
            tdu = (real)0;
        }
    }
    dl = inner ? tdl : (real)0;
    d = inner ? td : (real)1;
    du = inner ? tdu : (real)0;
    f = inner ? tf : (real)0;
}

// not-a-knot end value: c_e = c_1 (1 + r) - c_2 r, r = h_e / h_next
template <typename real>
__device__ __forceinline__ real nak_end(real c1, real c2, int h_e, int h_next)
{
    const real r = (real)h_e / (real)h_next;
    return c1 * ((real)1 + r) - c2 * r;
}

// x / y in the solve: IEEE division in FP64 (the oracle's arithmetic, bit
// for bit); in FP32 one hardware reciprocal (1 ulp) and a product
template <typename real>
__device__ __forceinline__ real sdiv(real x, real y)
{
    if constexpr (std::is_same<real, double>::value) return x / y;
    else return x * (real)__builtin_amdgcn_rcpf((float)y);
}

// Shuffles of the reduction by ST lanes: lane i gets lane i - ST (lane_up)
// or i + ST (lane_down); what a lane with no source gets is unspecified (the
// callers do not use it).  By one lane a DPP whole-wave shift (one vector
// move per 32 bits); farther a ds_bpermute.
template <int CTRL>
__device__ __forceinline__ int dpp_move(int v) { return __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, true); }
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) { return __int_as_float(dpp_move<CTRL>(__float_as_int(v))); }
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = dpp_move<CTRL>((int)b), hi = dpp_move<CTRL>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int ST, typename real>
__device__ __forceinline__ real lane_up(real v)
{
    if constexpr (ST == 1) return dpp_move<0x138>(v);
    else return shfl_up(v, ST);
}
template <int ST, typename real>
__device__ __forceinline__ real lane_down(real v)
{
    if constexpr (ST == 1) return dpp_move<0x130>(v);
    else return shfl_down(v, ST);
}

// 1 / x of a pivot.  FP64: the hardware's estimate, two Newton steps and the
// residual correction (correctly rounded, P. Markstein 1990); the operations
// of an IEEE division without those that scale and restore operands out of
// range.  Pivots are sums and differences of interval lengths, far inside it.
template <typename real>
__device__ __forceinline__ real pivot_inv(real x)
{
    if constexpr (std::is_same<real, double>::value) {
        double y = __builtin_amdgcn_rcp(x);
#pragma unroll
        for (int i = 0; i < 3; ++i) y = fma(fma(-x, y, 1.0), y, y);
        return y;
    } else {
        return sdiv<real>((real)1, x);
    }
}

// SYM: row g couples to row g + 1 as that to row g, or one of them not at all
// (true but for not-a-knot ends)
template <typename real, int B, bool SYM, class RowFn>
__device__ __forceinline__ void partition_pcr(int lane, RowFn row, real (&x)[B])
{
    real cp[B], al[B], be[B], ga[B];
#pragma unroll
    for (int q = 0; q <= B - 2; ++q) {
        real dl, d, du, f;
        row(q, dl, d, du, f);
        real inv;
        if (q == 0) {
            const real dl0 = (lane == 0) ? (real)0 : dl;
            inv = pivot_inv(d);
            al[0] = f * inv;
            be[0] = (-dl0) * inv;
        } else {
            inv = pivot_inv(d - dl * cp[q - 1]);
            al[q] = (f - dl * al[q - 1]) * inv;
            be[q] = (-dl) * be[q - 1] * inv;
        }
        cp[q] = du * inv;
        ga[q] = (q == B - 2) ? (-du) * inv : (real)0;
    }
#pragma unroll
    for (int q = B - 3; q >= 0; --q) {
        al[q] = al[q] - cp[q] * al[q + 1];
        be[q] = be[q] - cp[q] * be[q + 1];
        ga[q] = ga[q] - cp[q] * ga[q + 1];
    }
    // interface row q = B-1 -> reduced tridiagonal system in z_lane
    real dl, d, du, f;
    row(B - 1, dl, d, du, f);
    real na0 = lane_down<1>(al[0]), nb0 = lane_down<1>(be[0]), ng0 = lane_down<1>(ga[0]);
    if (lane == kWave - 1) {
        du = (real)0;
        na0 = (real)0;
        nb0 = (real)0;
        ng0 = (real)0;
    }
    real A = dl * be[B - 2];
    real D = (d + dl * ga[B - 2]) + du * nb0;
    real C = du * ng0;
    real R = (f - dl * al[B - 2]) - du * na0;
    // one reduction by st lanes; false if neither of its two terms changed any
    // D or R.  Then no later one does: with k1(l) = A(l) / D(l - st), unchanged
    // means |R(l - st) k1(l)| <= ulp / 2 of R(l) for every l, and the next
    // level's factor is k1(l - st) k1(l), so its products are smaller by another
    // factor of the unit roundoff (the same for D; a NaN counts as changed).
    // They are compared after each term, as two terms that cancel each other
    // need not be small; D only where that can happen: in a symmetric system
    // A(l) C(l - st) is a square or zero, and both terms reduce D.
    // Interfaces eight rows apart are coupled by about 0.27^8, so two or three
    // of the six levels do anything and one more shows it (a whole-stage pass
    // of 1000 FP64 samples 15.7 -> 14.6 thousand cycles, of 2800 FP32 ones 13.2
    // -> 12.1; the long series' solve launches -1 % FP32, -3 % FP64).
    auto level = [&](auto st_c) {
        constexpr int st = decltype(st_c)::value;
        const real Am = lane_up<st>(A), Dm = lane_up<st>(D), Cm = lane_up<st>(C),
                   Rm = lane_up<st>(R);
        const real Ap = lane_down<st>(A), Dp = lane_down<st>(D), Cp = lane_down<st>(C),
                   Rp = lane_down<st>(R);
        real a2 = (real)0, c2 = (real)0, d2 = D, r2 = R;
        if (lane - st >= 0) {
            const real k1 = sdiv<real>(A, Dm);
            a2 = -(Am * k1);
            d2 = d2 - Cm * k1;
            r2 = r2 - Rm * k1;
        }
        const real d1 = d2, r1 = r2;
        if (lane + st < kWave) {
            const real k2 = sdiv<real>(C, Dp);
            c2 = -(Cp * k2);
            d2 = d2 - Ap * k2;
            r2 = r2 - Rp * k2;
        }
        const bool changed =
            wave_ballot(!(SYM || d1 == D) | !(d2 == D) | !(r1 == R) | !(r2 == R)) != 0ull;
        A = a2;
        C = c2;
        D = d2;
        R = r2;
        return changed;
    };
    if (level(std::integral_constant<int, 1>{}) && level(std::integral_constant<int, 2>{}) &&
        level(std::integral_constant<int, 4>{}) && level(std::integral_constant<int, 8>{}) &&
        level(std::integral_constant<int, 16>{}))
        level(std::integral_constant<int, 32>{});
    const real z = sdiv<real>(R, D);
    real zl = lane_up<1>(z);
    if (lane == 0) zl = (real)0;
#pragma unroll
    for (int q = 0; q < B; ++q) x[q] = (q == B - 1) ? z : (al[q] + be[q] * zl) + ga[q] * z;
}

}  // namespace icm
