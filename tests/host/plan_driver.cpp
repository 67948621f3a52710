// Host code of the plan without a GPU (see fake_hip.cpp): one check per name
// on the command line; prints "ok" for each that holds.
#include "fake_hip.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../ceemdan-gpu_amd/csrc/icm_kernels.h"
#include "../../include/iceemdan_mi355x.h"

using namespace icm;

#define CHECK(x)                                                    \
    do {                                                            \
        if (!(x)) {                                                 \
            std::printf("line %d: %s\n", __LINE__, #x);             \
            return false;                                           \
        }                                                           \
    } while (0)

namespace {

struct Call {
    std::vector<int64_t> lens;
    std::vector<std::vector<double>> in, out;   // large enough for either dtype
    std::vector<void*> inp, outp;
    icm_config c;
    Call(std::vector<int64_t> l, int I, int M, int dtype, int stop = ICM_STOP_FIXED) : lens(std::move(l))
    {
        icm_config_default(&c);
        c.dtype = dtype;
        c.num_channels = (int)lens.size();
        c.lengths = lens.data();
        c.num_noise = I;
        c.num_imfs = M;
        c.stop_mode = stop;
        c.use_graph = 0;
        if (stop == ICM_STOP_RILLING) c.max_sifts = c.noise_max_sifts = 100;
        for (int64_t n : lens) {
            in.emplace_back(n, 1.0);
            out.emplace_back(n * M, 0.0);
        }
        for (auto& v : in) inp.push_back(v.data());
        for (auto& v : out) outp.push_back(v.data());
    }
};

int g_prefixes, g_stages, g_dirty;

bool is(const FakeLaunch& l, const char* kernel) { return std::strstr(l.name, kernel) != nullptr; }

// counts the launches of either path; a knot prefix whose control words are
// not clear is one that would write past the window list
void watch(const FakeLaunch& l)
{
    if (is(l, "k_stage")) ++g_stages;
    if (!is(l, "k_knot_prefix")) return;
    ++g_prefixes;
    const PassCtl pc = *(const PassCtl*)l.args[3];
    if (*pc.wincount != 0u || pc.dense[pc.epoch] != 0u) ++g_dirty;
}

void reset_watch()
{
    g_prefixes = g_stages = g_dirty = 0;
    fake_on_launch = watch;
}

// A staged forward that leaves the stage kernel between its calls.
bool staged_switch()
{
    for (int dtype : {ICM_DTYPE_F32, ICM_DTYPE_F64})
        for (int stop : {ICM_STOP_FIXED, ICM_STOP_RILLING})
            for (int how = 0; how < 3; ++how)
                for (int load = 0; load < 2; ++load) {
                    Call k({1000, 300}, 3, 4, dtype, stop);
                    icm_plan p = nullptr, q = nullptr;
                    reset_watch();
                    CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
                    CHECK(icm_forward_begin(p, k.inp.data(), nullptr, nullptr) == ICM_OK);
                    if (load) {
                        int64_t n = 0;
                        CHECK(icm_state_bytes(p, &n) == ICM_OK);
                        std::vector<char> state(n);
                        CHECK(icm_state_save(p, state.data(), n, nullptr) == ICM_OK);
                        CHECK(icm_plan_create(&k.c, &q) == ICM_OK);
                        CHECK(icm_state_load(q, state.data(), n, nullptr, nullptr) == ICM_OK);
                        std::swap(p, q);
                    }
                    CHECK(g_stages > 0 && g_prefixes == 0);
                    const int32_t cand[3] = {0, 0, 0};
                    if (how == 0) CHECK(icm_set_profiling(p, 1) == ICM_OK);
                    if (how == 1) CHECK(icm_set_tuning(p, ICM_PHASE_SIGNAL, cand, 3) == ICM_OK);
                    if (how == 2) CHECK(icm_set_trace(p, 2) == ICM_OK);
                    CHECK(icm_forward_stages(p, 3, nullptr, nullptr) == ICM_OK);
                    CHECK(g_prefixes > 0);
                    CHECK(g_dirty == 0);
                    CHECK(icm_forward_finish(p, k.outp.data(), nullptr) == ICM_OK);
                    CHECK(icm_plan_destroy(p) == ICM_OK);
                    if (q) CHECK(icm_plan_destroy(q) == ICM_OK);
                    CHECK(fake_used_bytes == 0);
                }
    return true;
}

// Launch shapes of the stage kernel at the most series a phase may have (2^28
// tiles): below 2^32 work-items, no scratch slot without a workgroup.
bool stage_grid()
{
    for (int size : {4, 8})
        for (int64_t ntl = 1; ntl <= 130; ++ntl)
            for (int64_t nser : {(int64_t)1, (int64_t)257, ((int64_t)1 << 28) / ntl}) {
                const StageGeom g = stage_geometry(size, 256 * ntl, nser);
                if (!g.ok) continue;
                CHECK(g.grid >= 1 && g.grid <= nser);
                CHECK((uint64_t)g.grid * g.nwv * 64 <= 0xFFFFFFFFull);
                CHECK(g.slot == 0 || g.slot * (uint64_t)g.grid <= (uint64_t)300 << 20);
            }
    return true;
}

// A plan stays within what icm_plan_bytes says and within ICM_MEMORY_BUDGET
// (but for its small tables, which the estimate leaves out), is refused where
// it was, and has the stage kernel's scratch where that fits.
bool budget()
{
    for (int dtype : {ICM_DTYPE_F32, ICM_DTYPE_F64})
        for (int n : {3000, 20000, 32768})
            for (int I : {20, 300}) {
                Call k({n, n - 7}, I, 3, dtype);
                setenv("ICM_WHOLE_STAGES", "0", 1);
                int64_t least = 0, most = 0;
                CHECK(icm_plan_bytes(&k.c, &least) == ICM_OK);
                setenv("ICM_WHOLE_STAGES", "1", 1);
                CHECK(icm_plan_bytes(&k.c, &most) == ICM_OK);
                const int64_t tables = (128 << 10) + least / 500;
                CHECK(n == 3000 ? most == least : most > least);
                for (int64_t room : {least - 1, least, (least + most) / 2, most + tables}) {
                    setenv("ICM_MEMORY_BUDGET", std::to_string(room).c_str(), 1);
                    icm_plan p = nullptr;
                    const int rc = icm_plan_create(&k.c, &p);
                    unsetenv("ICM_MEMORY_BUDGET");
                    CHECK(rc == (room < least ? ICM_ERR_OUT_OF_MEMORY : ICM_OK));
                    if (rc) continue;
                    CHECK(fake_used_bytes <= room + tables);
                    icm_plan_info info;
                    CHECK(icm_plan_get_info(p, &info) == ICM_OK);
                    CHECK(info.device_bytes <= fake_used_bytes && info.device_bytes >= fake_used_bytes - tables);
                    reset_watch();
                    CHECK(icm_set_autotune(p, 0) == ICM_OK);
                    CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
                    if (room > most) CHECK(g_stages > 0 && g_prefixes == 0);
                    CHECK(icm_plan_destroy(p) == ICM_OK);
                    CHECK(fake_used_bytes == 0);
                }
            }
    return true;
}

int64_t device_bytes(icm_plan p)
{
    icm_plan_info info;
    return icm_plan_get_info(p, &info) == ICM_OK ? info.device_bytes : -1;
}

// A backward whose buffers fit only in place of the stage kernel's scratch
// takes them there and counts them once.
bool backward_room()
{
    Call k({32768}, 40, 3, ICM_DTYPE_F64);
    for (int round = 0; round < 2; ++round) {
        icm_plan p = nullptr;
        CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        if (round) fake_free_bytes = fake_used_bytes + (30 << 20);
        const int rc = icm_backward(p, k.outp.data(), k.inp.data(), nullptr);
        fake_free_bytes = (long long)1 << 40;
        CHECK(rc == ICM_OK);
        // (pieces of an allocation begin at multiples of 256 bytes)
        CHECK(device_bytes(p) <= fake_used_bytes && device_bytes(p) >= fake_used_bytes - (64 << 10));
        CHECK(icm_plan_destroy(p) == ICM_OK);
        CHECK(fake_used_bytes == 0);
    }
    return true;
}

// The same for traces.
bool trace_room()
{
    Call k({32768}, 40, 3, ICM_DTYPE_F64);
    icm_plan p = nullptr;
    CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
    fake_free_bytes = fake_used_bytes + 1000;
    const int rc = icm_set_trace(p, 10);
    fake_free_bytes = (long long)1 << 40;
    CHECK(rc == ICM_OK);
    CHECK(device_bytes(p) <= fake_used_bytes && device_bytes(p) >= fake_used_bytes - (64 << 10));
    CHECK(icm_plan_destroy(p) == ICM_OK);
    CHECK(fake_used_bytes == 0);
    return true;
}

// The same for the records of a backward that sifts again: with room for the
// backward's buffers and not for the records, and for the records and not for
// their device table; then once more, with what it has.
bool record_room()
{
    Call k({32768}, 40, 3, ICM_DTYPE_F64);
    int64_t buffers = 0, records = 0;
    for (int keep = 1; keep >= 0; --keep) {
        icm_plan p = nullptr;
        k.c.keep_records = keep;   // with kept records the backward takes its buffers only
        CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        const long long before = fake_used_bytes;
        CHECK(icm_backward(p, k.outp.data(), k.inp.data(), nullptr) == ICM_OK);
        (keep ? buffers : records) = fake_used_bytes - before - (keep ? 0 : buffers);
        CHECK(icm_plan_destroy(p) == ICM_OK);
    }
    CHECK(buffers > 0 && records > 1 << 20);
    for (int64_t room : {buffers + 4096, buffers + records - 256}) {
        icm_plan p = nullptr;
        CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        fake_free_bytes = fake_used_bytes + room;
        reset_watch();
        for (int n = 0; n < 2; ++n) {
            const int rc = icm_backward(p, k.outp.data(), k.inp.data(), nullptr);
            if (rc != ICM_OK) fake_free_bytes = (long long)1 << 40;
            CHECK(rc == ICM_OK);
        }
        CHECK(g_prefixes > 0 && g_dirty == 0);   // without scratch: launches per step
        fake_free_bytes = (long long)1 << 40;
        reset_watch();
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        CHECK(icm_backward(p, k.outp.data(), k.inp.data(), nullptr) == ICM_OK);
        CHECK(g_stages == 0 && g_prefixes > 0 && g_dirty == 0);
        CHECK(device_bytes(p) <= fake_used_bytes && device_bytes(p) >= fake_used_bytes - (64 << 10));
        CHECK(icm_plan_destroy(p) == ICM_OK);
        CHECK(fake_used_bytes == 0);
    }
    return true;
}

// What icm_get_tuning returns of a plan with the default geometry can be given
// back without a change of path; a candidate moves its phase to sift launches
// until it is taken back.
bool tuning_round_trip()
{
    Call k({1000, 300}, 3, 4, ICM_DTYPE_F32);
    icm_plan p = nullptr;
    CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
    auto forward = [&] {
        reset_watch();
        return icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK;
    };
    int32_t v[2][3];
    for (int ph = 0; ph < 2; ++ph) CHECK(icm_get_tuning(p, ph, v[ph], 3) == ICM_OK);
    for (int ph = 0; ph < 2; ++ph) CHECK(icm_set_tuning(p, ph, v[ph], 3) == ICM_OK);
    CHECK(forward() && g_stages == 6 && g_prefixes == 0);
    const int32_t cand[3] = {-1, 2, -1};
    CHECK(icm_set_tuning(p, ICM_PHASE_SIGNAL, cand, 3) == ICM_OK);
    CHECK(forward() && g_stages == 3 && g_prefixes > 0);
    CHECK(icm_set_tuning(p, ICM_PHASE_SIGNAL, v[1], 3) == ICM_OK);
    CHECK(forward() && g_stages == 6 && g_prefixes == 0);
    CHECK(icm_set_tuning(p, ICM_PHASE_NOISE, cand, 3) == ICM_OK && icm_set_autotune(p, 0) == ICM_OK);
    CHECK(forward() && g_stages == 6 && g_prefixes == 0);
    CHECK(icm_plan_destroy(p) == ICM_OK);
    return true;
}

// Which path a plan takes by its series' length and number and its rows:
// both sides of the lines.
bool few_series()
{
    const int F = ICM_STOP_FIXED, R = ICM_STOP_RILLING;
    // (`more` channels of 300 samples beside the one)
    const struct { int dtype, stop, n, I, M; bool whole; int more; } t[] = {
        {ICM_DTYPE_F64, F, 32768, 4, 6, false},  {ICM_DTYPE_F64, F, 32768, 91, 6, false},
        {ICM_DTYPE_F64, F, 32768, 92, 6, true},  {ICM_DTYPE_F64, F, 28160, 65, 6, false},
        {ICM_DTYPE_F64, F, 28160, 66, 6, true},  {ICM_DTYPE_F64, F, 24064, 1, 6, false},
        {ICM_DTYPE_F64, F, 24064, 1, 7, true},   {ICM_DTYPE_F64, F, 14336, 1, 3, false},
        {ICM_DTYPE_F64, F, 14080, 1, 4, true},   {ICM_DTYPE_F64, F, 32768, 1, 12, true},
        {ICM_DTYPE_F64, R, 32768, 107, 6, false}, {ICM_DTYPE_F64, R, 32768, 108, 6, true},
        {ICM_DTYPE_F64, R, 24064, 4, 6, true},   {ICM_DTYPE_F32, F, 32768, 1, 4, false},
        {ICM_DTYPE_F32, F, 32768, 1, 5, true},   {ICM_DTYPE_F32, R, 32768, 1, 3, false},
        {ICM_DTYPE_F32, R, 32768, 1, 4, true},   {ICM_DTYPE_F64, F, 1000, 1, 2, true},
        {ICM_DTYPE_F64, F, 32768, 20, 6, false, 20}, {ICM_DTYPE_F64, F, 32768, 90, 6, true, 7},
        {ICM_DTYPE_F32, F, 32768, 20, 6, true, 20},
    };
    for (const auto& q : t) {
        std::vector<int64_t> lens(1 + q.more, 300);
        lens[0] = q.n;
        Call k(lens, q.I, q.M, q.dtype, q.stop);
        icm_plan p = nullptr;
        CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
        int left = -1;
        CHECK(icm_get_tuning_left(p, &left) == ICM_OK && left == 0);
        reset_watch();
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        if ((g_stages > 0) != q.whole || (g_prefixes > 0) == q.whole)
            std::printf("dtype %d stop %d %d x %d M %d\n", q.dtype, q.stop, q.I, q.n, q.M);
        CHECK((g_stages > 0) == q.whole && (g_prefixes > 0) != q.whole);
        CHECK(icm_plan_destroy(p) == ICM_OK);
    }
    return true;
}

// The same for more than 128 series; the launches per step are tuned then.
bool few_rows()
{
    const struct { int dtype, stop, n, I, M; bool whole; } t[] = {
        {ICM_DTYPE_F64, ICM_STOP_FIXED, 32768, 300, 7, false}, {ICM_DTYPE_F64, ICM_STOP_FIXED, 32768, 300, 8, true},
        {ICM_DTYPE_F64, ICM_STOP_FIXED, 32768, 256, 5, true},   {ICM_DTYPE_F64, ICM_STOP_FIXED, 32768, 256, 4, false},
        {ICM_DTYPE_F64, ICM_STOP_FIXED, 24576, 300, 5, false},
        {ICM_DTYPE_F64, ICM_STOP_FIXED, 24576, 300, 6, true},   {ICM_DTYPE_F64, ICM_STOP_FIXED, 24064, 300, 3, true},
        {ICM_DTYPE_F64, ICM_STOP_RILLING, 28160, 300, 4, false}, {ICM_DTYPE_F64, ICM_STOP_RILLING, 28160, 300, 5, true},
        {ICM_DTYPE_F32, ICM_STOP_FIXED, 32768, 300, 3, true},
    };
    for (const auto& q : t) {
        Call k({q.n}, q.I, q.M, q.dtype, q.stop);
        icm_plan p = nullptr;
        CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
        int left = -1;
        CHECK(icm_get_tuning_left(p, &left) == ICM_OK && (left == 0) == q.whole);
        reset_watch();
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        if ((g_stages > 0) != q.whole) std::printf("dtype %d stop %d %d x %d M %d\n", q.dtype, q.stop, q.I, q.n, q.M);
        CHECK((g_stages > 0) == q.whole && (g_prefixes > 0) != q.whole);
        CHECK(icm_plan_destroy(p) == ICM_OK);
    }
    return true;
}

int g_past, g_through;

void watch_sift(const FakeLaunch& l)
{
    if (!is(l, "k_sift_w")) return;
    const bool f64 = is(l, "k_sift_wId");
    const bool past = f64 ? ((const SiftArgs<double>*)l.args[0])->past_caches
                          : ((const SiftArgs<float>*)l.args[0])->past_caches;
    ++(past ? g_past : g_through);
}

// Samples go past the caches where a phase's two buffers exceed 256 MB, each
// phase by its own size.
bool past_caches()
{
    const struct { int dtype, I, channels, past, through; } t[] = {
        {ICM_DTYPE_F64, 68, 1, 0, 2}, {ICM_DTYPE_F64, 69, 1, 2, 0}, {ICM_DTYPE_F64, 35, 2, 1, 1},
        {ICM_DTYPE_F32, 137, 1, 0, 2}, {ICM_DTYPE_F32, 138, 1, 2, 0},
    };
    for (const auto& q : t) {
        Call k(std::vector<int64_t>(q.channels, 244032), q.I, 2, q.dtype);
        k.c.max_sifts = k.c.noise_max_sifts = 1;
        icm_plan p = nullptr;
        CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
        CHECK(icm_set_autotune(p, 0) == ICM_OK);
        g_past = g_through = 0;
        fake_on_launch = watch_sift;
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        CHECK(g_past == q.past && g_through == q.through);
        CHECK(icm_plan_destroy(p) == ICM_OK);
    }
    return true;
}

std::vector<FakeLaunch> g_noise;
std::vector<std::vector<int>> g_noise_len;

void watch_noise(const FakeLaunch& l)
{
    if (!is(l, "k_noise")) return;
    const int* len = *(const int**)l.args[1];
    g_noise.push_back(l);
    g_noise_len.emplace_back(len, len + l.grid.z);
}

// Noise of a plan of very uneven lengths: every length once, by workgroups
// enough, and at most as many again that only find themselves past an end.
bool noise_groups()
{
    const int I = 20;
    for (int kind = 0; kind < 3; ++kind) {
        std::vector<int64_t> lens;
        for (int c = 0; c < 300; ++c) lens.push_back(256 + c);
        if (kind == 1) lens[150] = 1 << 20;
        if (kind == 2)
            for (int c = 0; c < 300; c += 3) lens[c] = 5000 + 401 * c;
        Call k(lens, I, 2, ICM_DTYPE_F32);
        k.c.max_sifts = k.c.noise_max_sifts = 1;
        icm_plan p = nullptr;
        CHECK(icm_plan_create(&k.c, &p) == ICM_OK);
        g_noise.clear();
        g_noise_len.clear();
        fake_on_launch = watch_noise;
        CHECK(icm_forward(p, k.inp.data(), k.outp.data(), nullptr, nullptr) == ICM_OK);
        CHECK(icm_plan_destroy(p) == ICM_OK);
        std::vector<int64_t> seen;
        int64_t needed = 0, launched = 0;
        for (int64_t n : lens) needed += I * ((n + 1023) / 1024);
        for (size_t q = 0; q < g_noise.size(); ++q) {
            launched += (int64_t)g_noise[q].grid.x * g_noise[q].grid.y * g_noise[q].grid.z;
            for (int n : g_noise_len[q]) {
                seen.push_back(n);
                CHECK((int64_t)g_noise[q].grid.x * 1024 >= n && g_noise[q].grid.y == I);
            }
        }
        CHECK(seen == lens);
        CHECK(launched <= 2 * needed);
        CHECK(kind != 0 || g_noise.size() == 1);
    }
    return true;
}

}  // namespace

int main(int argc, char** argv)
{
    const struct { const char* name; bool (*run)(); } all[] = {
        {"staged_switch", staged_switch},
        {"stage_grid", stage_grid},
        {"budget", budget},
        {"backward_room", backward_room},
        {"record_room", record_room},
        {"trace_room", trace_room},
        {"tuning_round_trip", tuning_round_trip},
        {"few_series", few_series},
        {"few_rows", few_rows},
        {"noise_groups", noise_groups},
        {"past_caches", past_caches},
    };
    for (int i = 1; i < argc; ++i)
        for (const auto& t : all)
            if (!std::strcmp(argv[i], t.name) && t.run()) std::printf("%s ok\n", t.name);
    return 0;
}
