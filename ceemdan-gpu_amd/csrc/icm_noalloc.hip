// One sift pass over equal-length series (icm_sift_pass and
// icm_sift_pass_static).
//
// Series whose knot rows fit LDS take the stage kernel: one launch, no other
// memory.  Longer ones take the launch-per-step kernels on buffers carved
// from one piece of device memory: icm_sift_pass allocates it for the call;
// icm_sift_pass_static, for callers that may not allocate (tight serving
// loops, harnesses that forbid it), uses one file-scope device array
// `scratch` of kScratchBytes (each GPU the library runs on holds its own copy
// until the process ends).  The series tables of the I equal-length series
// are written on the device by a kernel (closed form), and every control word
// is cleared by a fill kernel, so no host-to-device copy is made either.
// (A plan built for the one pass took 3.3 ms at 200 x 30504 FP32, nearly all
// of it allocations and table copies.)
//
// Limits of icm_sift_pass_static: I * N <= kMaxSamples (2^21) and I <=
// kMaxSeries (4096); larger calls return ICM_ERR_INVALID_ARG.  All calls on
// one GPU share that GPU's array and it keeps the last call's contents: two
// calls that overlap on one GPU (other threads, other streams) race and must
// be serialised by the caller.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "../../include/iceemdan_mi355x.h"
#include "icm_errors.h"
#include "icm_kernels.h"

namespace icm {
namespace {

constexpr int64_t kMaxSamples = (int64_t)1 << 21;
constexpr int kMaxSeries = 4096;
constexpr int kTile = 256;         // samples per tile of the tile kernels
// windowed solve: halo rows per side (FP32 16, FP64 32) and rows kept per
// window, as the plans use them
template <typename real>
constexpr int solve_h() { return std::is_same<real, float>::value ? 16 : 32; }
template <typename real>
constexpr int solve_k() { return 64 * 8 - 2 * solve_h<real>(); }
constexpr size_t kScratchBytes = (size_t)24 << 20;

__device__ __align__(256) unsigned char scratch[kScratchBytes];

// device address of `scratch` per device (hipGetSymbolAddress, once each)
std::mutex g_mu;
void* g_ptr[64] = {};

int scratch_ptr(void** out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return ICM_ERR_HIP;
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return ICM_ERR_HIP;
        g_ptr[dev] = p;
    }
    *out = g_ptr[dev];
    return ICM_OK;
}

// Tables of I series of N samples each, back to back (closed form), and
// the segments of `seg` tiles, one wavefront each in the sift.
__global__ void k_uniform_series(int I, int N, int ntl, int seg, int nseg_s, int* tile_series,
                                 int* tile0, int* ntl_out, int* len, int* chan, int* nidx,
                                 int64_t* off, int64_t* kbase, int64_t* eoff, Segment* segs)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t ntiles = (int64_t)I * ntl;
    if (i < ntiles) tile_series[i] = (int)(i / ntl);
    if (i < I) {
        tile0[i] = (int)(i * ntl);
        ntl_out[i] = ntl;
        len[i] = N;
        chan[i] = 0;
        nidx[i] = (int)i;
        off[i] = i * N;
        kbase[i] = i * (int64_t)(N / 2 + 2);
        eoff[i] = i * N;
    }
    if (i < (int64_t)I * nseg_s) {
        Segment g;
        g.s = (int)(i / nseg_s);
        g.t_first = (int)(i % nseg_s) * seg;
        g.count = std::min(seg, ntl - g.t_first);
        g.pad = 0;
        segs[i] = g;
    }
}

// bump allocator over one piece of memory (256-byte aligned pieces); with a
// null base it only adds up
struct Carve {
    char* base;
    size_t used = 0;
    template <typename T>
    T* take(int64_t n)
    {
        used = (used + 255) & ~(size_t)255;
        T* p = base ? (T*)(base + used) : nullptr;
        used += (size_t)std::max<int64_t>(n, 1) * sizeof(T);
        return p;
    }
};

template <typename real>
struct Tables {
    int ntl, ntiles, seg, nseg_s;
    int64_t kstride;
    int *tile_series, *tile0, *ntlv, *len, *chan, *nidx;
    int64_t *off, *kbase, *eoff;
    Segment* segs;
    KnotsDev<real> k;
    real* c;
    int* winlist;
    unsigned* ctlw;
    void take(Carve& cv, int N, int I)
    {
        ntl = (N + kTile - 1) / kTile;
        ntiles = I * ntl;
        seg = std::max(1, std::min(32, ntiles / 56000));
        nseg_s = (ntl + seg - 1) / seg;
        const int64_t kcap = N / 2 + 2;
        kstride = (int64_t)I * kcap;
        const int64_t maxwin = (int64_t)I * 2 * ((kcap + solve_k<real>() - 1) / solve_k<real>());
        tile_series = cv.take<int>(ntiles);
        tile0 = cv.take<int>(I);
        ntlv = cv.take<int>(I);
        len = cv.take<int>(I);
        chan = cv.take<int>(I);
        nidx = cv.take<int>(I);
        off = cv.take<int64_t>(I);
        kbase = cv.take<int64_t>(I);
        eoff = cv.take<int64_t>(I);
        segs = cv.take<Segment>((int64_t)I * nseg_s);
        k = KnotsDev<real>{};
        k.cnt = cv.take<int>(2 * (int64_t)ntiles);
        k.pre = cv.take<int>(2 * (int64_t)ntiles);
        k.n = cv.take<int>(2 * (int64_t)I);
        k.fix = cv.take<real>(4 * (int64_t)I);
        k.nbx = cv.take<int>(6 * (int64_t)ntiles);
        k.nby = cv.take<real>(6 * (int64_t)ntiles);
        k.mask = cv.take<uint64_t>(8 * (int64_t)ntiles);
        c = cv.take<real>(2 * kstride);
        winlist = cv.take<int>(kWinItem * maxwin);
        // control words: [0..3] window counts, [4..7] over-full counts,
        // [12] error word (epochs 1 and 2 are used)
        ctlw = cv.take<unsigned>(16);
    }
};

// the launch-per-step kernels on the carved tables
template <typename real>
int sift_steps(const Tables<real>& t, const real* h, int N, int I, real* h_new, int32_t* d_nk,
               hipStream_t st)
{
    const int ntl = t.ntl, ntiles = t.ntiles, seg = t.seg, nseg_s = t.nseg_s;
    const KnotsDev<real>& k = t.k;
    unsigned* ctlw = t.ctlw;

    hipError_t e;
    const int64_t items = std::max<int64_t>(ntiles, (int64_t)I * nseg_s);
    hipLaunchKernelGGL(k_uniform_series, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, st,
                       I, N, ntl, seg, nseg_s, t.tile_series, t.tile0, t.ntlv, t.len, t.chan, t.nidx,
                       t.off, t.kbase, t.eoff, t.segs);
    if ((e = hipGetLastError()) != hipSuccess) return ICM_ERR_HIP;
    if ((e = launch_fill_u32(ctlw, 0u, 16, st)) != hipSuccess) return ICM_ERR_HIP;

    SeriesDev sd{};
    sd.tile_series = t.tile_series;
    sd.tile0 = t.tile0;
    sd.ntl = t.ntlv;
    sd.off = t.off;
    sd.len = t.len;
    sd.kbase = t.kbase;
    sd.chan = t.chan;
    sd.eoff = t.eoff;
    sd.nidx = t.nidx;
    sd.nseries = I;
    sd.ntiles = ntiles;
    sd.max_tiles = ntl;
    sd.kstride = t.kstride;
    sd.cap = kTile / 2 + 2;
    int* err = (int*)(ctlw + 12);
    auto ctl = [&](uint32_t epoch) {
        PassCtl pc{};
        pc.epoch = epoch;
        pc.winlist = t.winlist;
        pc.wincount = ctlw + epoch;
        pc.K = solve_k<real>();
        pc.H = solve_h<real>();
        pc.err = err;
        pc.dense = ctlw + 4;
        pc.run = nullptr;
        return pc;
    };
    // knots of the input (no copy of its samples), prefixes, windows
    InitArgs<real> ia{};
    ia.mode = INIT_KNOTS;
    ia.src = h;
    if (launch_init<real>(sd, ia, nullptr, k, ctl(1), st) != hipSuccess) return ICM_ERR_HIP;
    if (launch_knot_prefix<real>(sd, k, h, ctl(1), nullptr, st) != hipSuccess) return ICM_ERR_HIP;
    SolveArgs<real> sa{};
    sa.sd = sd;
    sa.k = k;
    sa.h = h;
    sa.c = t.c;
    sa.winlist = t.winlist;
    sa.wincount = ctlw + 1;
    sa.err = err;
    if (launch_solve<real>(sa, 4096, st) != hipSuccess) return ICM_ERR_HIP;
    SiftArgs<real> a{};
    a.sd = sd;
    a.segs = t.segs;
    a.h_in = h;
    a.h_out = h_new;
    a.kin = k;
    a.c = t.c;
    a.kout = k;
    a.emit = 0;
    a.pc = ctl(2);
    a.queue = nullptr;   // one wavefront per segment (the grid is small here)
    a.past_caches = sift_past_caches((int64_t)I * N, sizeof(real));
    if (launch_sift<real>(a, I * nseg_s, st) != hipSuccess) return ICM_ERR_HIP;
    if (d_nk && launch_copy<float>((float*)d_nk, (const float*)k.n, 2 * (int64_t)I, st) != hipSuccess)
        return ICM_ERR_HIP;
    int h_err = 0;
    if (hipMemcpyAsync(&h_err, err, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return ICM_ERR_HIP;
    return h_err ? ICM_ERR_DEVICE : ICM_OK;
}

// The stage kernel, where the series' knot rows fit LDS; false: they do not.
template <typename real>
bool sift_whole(const real* h, int N, int I, real* h_new, int32_t* d_nk, hipStream_t st, int& rc)
{
    const StageGeom g = stage_geometry((int)sizeof(real), N, I);
    if (!g.ok || g.slot) return false;
    StageArgs<real> a{};
    a.uniform_len = N;
    a.nseries = I;
    a.ia.mode = INIT_KNOTS;
    a.ia.src = h;
    a.hA = a.hB = a.out = h_new;
    a.passes = 1;
    a.need_out = 1;
    a.nk_out = d_nk;
    rc = launch_stage<real>(a, g, st) == hipSuccess && hipStreamSynchronize(st) == hipSuccess
             ? ICM_OK
             : ICM_ERR_HIP;
    return true;
}

template <typename real>
int sift_alloc(const real* h, int N, int I, real* h_new, int32_t* d_nk, hipStream_t st)
{
    // an output over the input (in place, or any overlap) gets a copy of it
    const int64_t n = (int64_t)N * I;
    const bool overlap = h < h_new + n && h_new < h + n;
    int rc = ICM_OK;
    if (!overlap && sift_whole<real>(h, N, I, h_new, d_nk, st, rc)) return rc;
    Tables<real> t;
    auto take = [&](Carve& cv) {
        t.take(cv, N, I);
        return overlap ? cv.take<real>(n) : nullptr;
    };
    Carve size{nullptr}, cv{nullptr};
    (void)take(size);
    if (hipMalloc((void**)&cv.base, size.used) != hipSuccess) {
        (void)hipGetLastError();
        return ICM_ERR_OUT_OF_MEMORY;
    }
    real* copy = take(cv);
    if (overlap && launch_copy<real>(copy, h, n, st) != hipSuccess) rc = ICM_ERR_HIP;
    if (rc == ICM_OK) rc = sift_steps<real>(t, overlap ? copy : h, N, I, h_new, d_nk, st);
    if (hipFree(cv.base) != hipSuccess && rc == ICM_OK) rc = ICM_ERR_HIP;
    return rc;
}

template <typename real>
int sift_static(const real* h, int N, int I, real* h_new, int32_t* d_nk, hipStream_t st)
{
    Carve size{nullptr};
    Tables<real> t;
    t.take(size, N, I);
    if (size.used > kScratchBytes) return ICM_ERR_INVALID_ARG;
    int rc = ICM_OK;
    if (sift_whole<real>(h, N, I, h_new, d_nk, st, rc)) return rc;
    void* base = nullptr;
    if ((rc = scratch_ptr(&base))) return rc;
    Carve cv{(char*)base};
    t.take(cv, N, I);
    return sift_steps<real>(t, h, N, I, h_new, d_nk, st);
}

}  // namespace

int sift_uniform(int dtype, const void* h, int64_t N, int64_t I, void* h_new, int32_t* nk,
                 hipStream_t st)
{
    if (dtype == ICM_DTYPE_F64)
        return sift_alloc<double>((const double*)h, (int)N, (int)I, (double*)h_new, nk, st);
    return sift_alloc<float>((const float*)h, (int)N, (int)I, (float*)h_new, nk, st);
}
}  // namespace icm

extern "C" int icm_sift_pass_static(int dtype, const void* d_h, int64_t N, int64_t I,
                                    void* d_h_new, int32_t* d_nk, void* stream)
{
    if (!d_h || !d_h_new || N < 4 || N > 16000000 || I < 1 || I > icm::kMaxSeries ||
        N * I > icm::kMaxSamples)
        return ICM_ERR_INVALID_ARG;
    if (dtype == ICM_DTYPE_F64)
        return icm::sift_static<double>((const double*)d_h, (int)N, (int)I, (double*)d_h_new, d_nk,
                                        (hipStream_t)stream);
    if (dtype == ICM_DTYPE_F32)
        return icm::sift_static<float>((const float*)d_h, (int)N, (int)I, (float*)d_h_new, d_nk,
                                       (hipStream_t)stream);
    return ICM_ERR_INVALID_ARG;
}
