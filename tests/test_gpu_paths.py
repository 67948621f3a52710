"""The two forward paths against each other with the path forced by
ICM_WHOLE_STAGES when the plan is made (0: launches per step, 1: whole stages
in one workgroup wherever the series' length allows), and each against the
oracle where the other tests' plans no longer reach it."""
import importlib
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")
STEPS, STAGES = "0", "1"


def _sig():
    return importlib.import_module("ceemdan-gpu_amd.signals")


def _inputs(dtype, lens):
    import torch
    out = []
    for c, n in enumerate(lens):
        x = _sig().eeg_like(n, seed=500 + c) if n >= 64 else np.random.default_rng(n).standard_normal(n)
        out.append(torch.tensor(x, dtype=dtype, device="cuda"))
    return out


def _same(a, b):
    import torch
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    assert torch.equal(torch.isnan(a), torch.isnan(b))


def _plan(icm, monkeypatch, path, lens, I, M, **kw):
    """A plan on the given path, and that it took it: a plan of the launches
    per step has sift geometries to tune, one of whole stages none (the tuning
    is then switched off)."""
    monkeypatch.setenv("ICM_WHOLE_STAGES", path)
    plan = icm.Plan(lens, I, M, **kw)
    monkeypatch.delenv("ICM_WHOLE_STAGES")
    assert (plan.tuning_left() > 0) == (path == STEPS)
    plan.set_autotune(0)
    return plan


# (lengths, realizations): the shapes of a workgroup with one series each (one
# tile, tile and wave edges, one tile per wave, several), the longest it takes,
# and more series than workgroups: 300 of 3000 and 270 x 2 of uneven length
# take 8 waves of several tiles in FP32, 300 of 4700 and 9100 and 260 of 16384 the
# scratch slots of a workgroup one after the other
PATHS = [([4, 5, 63], 3), ([255, 256, 257, 1000], 3), ([1025, 3000, 4096], 3), ([4097, 4700], 3),
         ([8192, 9100], 3), ([16384, 16383], 3), ([30504, 5], 3), ([32768], 3), ([3000], 300),
         ([2049, 3583], 270), ([4700], 300), ([9100, 4801], 150), ([16384], 260)]


@pytest.mark.parametrize("lens,I", PATHS, ids=lambda v: "-".join(map(str, v)) if isinstance(v, list) else str(v))
@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("stop,nak", [(0, 0), (0, 1), (1, 0)])
def test_both_paths_compute_the_same_bits(icm, dev, monkeypatch, lens, I, dt, stop, nak):
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    M, S = 3, 5
    print(f"case: paths {dt} stop={stop} nak={nak} lens={lens} I={I}", flush=True)
    xs = _inputs(dtype, lens)
    got = []
    for path in (STEPS, STAGES):
        plan = _plan(icm, monkeypatch, path, lens, I, M, dtype=dtype, stop_mode=stop, max_sifts=S,
                     boundary=nak, noise_max_sifts=S if stop == 0 else 40, use_graph=False, device=dev)
        got.append([o.clone() for o in plan.forward(xs)] + [plan.noise_modes()])
        plan.close()
    for a, b in zip(*got):
        _same(a, b)


@pytest.mark.parametrize("lens,I", [([300, 4096], 3), ([32768], 3), ([3000], 300), ([4700, 4801], 150),
                                    ([16384], 260)],
                         ids=lambda v: "-".join(map(str, v)) if isinstance(v, list) else str(v))
@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("keep", [True, False])
def test_records_of_both_paths_give_the_same_gradient(icm, dev, monkeypatch, lens, I, dt, keep):
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    M, S = 3, 5
    print(f"case: records {dt} keep={keep} lens={lens} I={I}", flush=True)
    xs = _inputs(dtype, lens)
    rng = np.random.default_rng(3)
    gs = [torch.tensor(rng.standard_normal((M, n)), dtype=dtype, device="cuda") for n in lens]
    got = []
    for path in (STEPS, STAGES):
        plan = _plan(icm, monkeypatch, path, lens, I, M, dtype=dtype, max_sifts=S, use_graph=False,
                     device=dev, keep_records=keep)
        plan.forward(xs)
        got.append([g.clone() for g in plan.backward(gs)])
        plan.close()
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_more_series_than_workgroups(icm, dev, monkeypatch):
    """17 x 65535 series of 8 samples: more than the stage kernel's largest
    grid, each workgroup of four waves takes one or two."""
    import torch
    lens, I, M = [8] * 17, 65535, 2
    print("case: 1114095 series", flush=True)
    xs = _inputs(torch.float32, lens)
    got = []
    for path in (STEPS, STAGES):
        plan = _plan(icm, monkeypatch, path, lens, I, M, dtype=torch.float32, max_sifts=2,
                     use_graph=False, device=dev)
        got.append([o.clone() for o in plan.forward(xs)])
        plan.close()
    for a, b in zip(*got):
        _same(a, b)


@pytest.mark.parametrize("keep", [True, False])
def test_phases_on_different_paths(icm, dev, monkeypatch, keep):
    """4 x 32768, I = 23, M = 6 in FP64: 23 noise-mode series launch step by step,
    beside 92 series of the CEEMDAN phase in whole stages; replayed with other
    inputs, forward and adjoint, and equal to launches per step."""
    import torch
    lens, I, M, S = [32768] * 4, 23, 6, 5
    print(f"case: phases on different paths keep={keep}", flush=True)
    kw = dict(dtype=torch.float64, max_sifts=S, device=dev, keep_records=keep)
    steps = _plan(icm, monkeypatch, STEPS, lens, I, M, use_graph=False, **kw)
    monkeypatch.delenv("ICM_WHOLE_STAGES", raising=False)
    plan = icm.Plan(lens, I, M, **kw)
    assert plan.tuning_left() == 0
    rng = np.random.default_rng(8)
    for seed in range(4):
        xs = [torch.tensor(_sig().eeg_like(n, seed=900 + 10 * seed + c), device=dev)
              for c, n in enumerate(lens)]
        gs = [torch.tensor(rng.standard_normal((M, n)), device=dev) for n in lens]
        for a, b in zip(plan.forward(xs) + plan.backward(gs), steps.forward(xs) + steps.backward(gs)):
            _same(a, b)
    assert plan.graph_status() == 1
    plan.close()
    steps.close()


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("stop", [0, 1])
def test_staged_forward_that_changes_path(icm, dev, monkeypatch, dt, stop):
    """A staged forward whose stages are profiled, tuned or traced in part
    gives icm_forward's bits."""
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    lens, I, M = [3000, 700], 4, 5
    print(f"case: staged path change {dt} stop={stop}", flush=True)
    xs = _inputs(dtype, lens)
    kw = dict(dtype=dtype, stop_mode=stop, max_sifts=6, noise_max_sifts=6 if stop == 0 else 40,
              device=dev)
    plan = _plan(icm, monkeypatch, STAGES, lens, I, M, **kw)
    ref = [o.clone() for o in plan.forward(xs)]
    plan.close()

    def profile(p, on):
        icm._check(icm.lib().icm_set_profiling(p._h, 1 if on else 0))

    def tune(p, on):
        p.set_tuning(icm.PHASE_SIGNAL, [2 if on else -1] * (M - 1))

    def trace(p, on):
        p.set_trace(3 if on else 0)

    for change in (profile, tune, trace):
        plan = _plan(icm, monkeypatch, STAGES, lens, I, M, **kw)
        for _ in range(2):
            plan.forward_begin(xs)
            plan.forward_stages(1)
            change(plan, True)
            plan.forward_stages(1)
            state = plan.save_state()
            change(plan, False)
            plan.forward_stages(1)
            change(plan, True)
            plan.forward_stages(M)
            for a, b in zip(plan.forward_finish(), ref):
                _same(a, b)
            change(plan, False)
            assert plan.load_state(state) == 2
            change(plan, True)
            plan.forward_stages(M)
            for a, b in zip(plan.forward_finish(), ref):
                _same(a, b)
            change(plan, False)
            for a, b in zip(plan.forward(xs), ref):   # captured on the stage path
                _same(a, b)
        plan.close()


@pytest.mark.parametrize("sparse_stage,dense_max,stop", [(0, 1 << 30, 0), (0, 1 << 30, 1), (0, 0, 0),
                                                         (0, 0, 1), (0, 20, 0), (1, -1, 0)])
@pytest.mark.parametrize("segment", ["1", "3", "8"])
def test_over_full_tiles_in_segments(icm, orc, dev, monkeypatch, sparse_stage, dense_max, stop, segment):
    """Sift launches with small knot tables over 79 tiles, most of them
    over-full in the first stages: the tile after one of them evaluates its
    left neighbour itself, the one before closes its own last sample, and
    passes with more of them than tolerated run with full tables.  The oracle's
    bits, FIXED and RILLING, segments of 1, 3 and 8 tiles."""
    import torch
    monkeypatch.setenv("ICM_SPARSE_STAGE", str(sparse_stage))
    monkeypatch.setenv("ICM_SPARSE_DENSE_MAX", str(dense_max))
    monkeypatch.setenv("ICM_SEGMENT_TILES", segment)
    N, I, M = 20000, 4, 4
    x = _sig().eeg_like(N, seed=3)
    print(f"case: over-full tiles stage={sparse_stage} dense={dense_max} stop={stop} seg={segment}", flush=True)
    S = 8 if stop == 0 else 40
    cap = S if stop == 0 else 100
    w = icm.noise(I, N, seed=21, dtype=torch.float64, device=dev)
    ref = orc.iceemdan(x, w.cpu().numpy(), M, stop_mode=stop, S_or_cap=S, noise_cap=cap)["imfs"]
    plan = _plan(icm, monkeypatch, STEPS, [N], I, M, dtype=torch.float64, stop_mode=stop, max_sifts=S,
                 noise_max_sifts=cap, use_graph=False, device=dev)
    got = plan.forward([torch.tensor(x, device=dev)], noise=w)[0].cpu().numpy()
    plan.close()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("sparse_stage,dense_max,stop", [(0, 1 << 30, 0), (0, 1 << 30, 1), (0, 20, 0)])
def test_over_full_tiles_in_segments_fp32(icm, dev, monkeypatch, sparse_stage, dense_max, stop):
    """The same in FP32, with quads: the bits of full tables everywhere."""
    import torch
    lens, I, M = [20000, 20001, 19903], 4, 4
    print(f"case: over-full tiles f32 stage={sparse_stage} dense={dense_max} stop={stop}", flush=True)
    xs = _inputs(torch.float32, lens)
    got = []
    for stage, dense, segment in ((M, 0, "1"), (sparse_stage, dense_max, "3"), (sparse_stage, dense_max, "8")):
        monkeypatch.setenv("ICM_SPARSE_STAGE", str(stage))
        monkeypatch.setenv("ICM_SPARSE_DENSE_MAX", str(dense))
        monkeypatch.setenv("ICM_SEGMENT_TILES", segment)
        plan = _plan(icm, monkeypatch, STEPS, lens, I, M, dtype=torch.float32, stop_mode=stop, max_sifts=8,
                     noise_max_sifts=8 if stop == 0 else 60, use_graph=False, device=dev)
        got.append([o.clone() for o in plan.forward(xs)] + [plan.noise_modes()])
        plan.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            _same(a, b)


@pytest.mark.parametrize("N", [9000, 29000])
@pytest.mark.parametrize("stop", [0, 1])
def test_one_wave_prefix_against_the_oracle(icm, orc, dev, monkeypatch, N, stop):
    """k_knot_prefix_w with one and two chunks of 64 tiles per series."""
    import torch
    I, M = 3, 4
    x = _sig().eeg_like(N, seed=31)
    print(f"case: one-wave prefix N={N} stop={stop}", flush=True)
    S = 8 if stop == 0 else 40
    cap = S if stop == 0 else 100
    w = icm.noise(I, N, seed=22, dtype=torch.float64, device=dev)
    ref = orc.iceemdan(x, w.cpu().numpy(), M, stop_mode=stop, S_or_cap=S, noise_cap=cap)["imfs"]
    plan = _plan(icm, monkeypatch, STEPS, [N], I, M, dtype=torch.float64, stop_mode=stop, max_sifts=S,
                 noise_max_sifts=cap, use_graph=False, device=dev)
    got = plan.forward([torch.tensor(x, device=dev)], noise=w)[0].cpu().numpy()
    plan.close()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("rows,n", [(3, 4), (5, 257), (2, 4600), (2, 4700), (2, 30504), (1, 70001)])
def test_allocation_free_pass_in_place(icm, dev, dt, rows, n):
    """icm_sift_pass_static with its output over its input."""
    import ctypes as C

    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    print(f"case: static in place {dt} {rows} x {n}", flush=True)
    h = torch.tensor(np.random.default_rng(n).standard_normal((rows, n)), dtype=dtype, device="cuda")
    ref, nk = icm.sift_pass(h)
    k2 = torch.zeros_like(nk)
    st = C.c_void_p(torch.cuda.current_stream(h.device).cuda_stream)
    assert icm.lib().icm_sift_pass_static(icm._dtype_code(dtype), C.c_void_p(h.data_ptr()), n, rows,
                                          C.c_void_p(h.data_ptr()), C.c_void_p(k2.data_ptr()), st) == 0
    assert torch.equal(h, ref) and torch.equal(k2, nk)


@pytest.mark.parametrize("dt,C", [("f64", 8), ("f32", 16)])
@pytest.mark.parametrize("stop", [0, 1])
def test_samples_past_the_caches(icm, dev, dt, C, stop):
    """8 x 70 k FP64 (16 FP32) channels, I = 32: 143 MB a buffer, sifted past the
    caches; each of two channels alone, 18 (9) MB, through them.  The same bits."""
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    lens, I, M = [70001 - 3 * c for c in range(C)], 32, 3
    print(f"case: past the caches {dt} stop={stop}", flush=True)
    kw = dict(dtype=dtype, stop_mode=stop, max_sifts=4 if stop == 0 else 12,
              noise_max_sifts=4 if stop == 0 else 20, use_graph=False, device=dev)
    xs = _inputs(dtype, lens)
    plan = icm.Plan(lens, I, M, **kw)
    assert plan.info()["signal_samples"] * xs[0].element_size() > 128 << 20
    got = [o.clone() for o in plan.forward(xs)]
    plan.close()
    for c in (0, C - 1):
        alone = icm.Plan([lens[c]], I, M, **kw)
        _same(alone.forward([xs[c]])[0], got[c])
        alone.close()
