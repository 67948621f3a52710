"""Whole stages of short series in one workgroup against the launch-per-step
path: the same bits, for lengths at the edges of tiles, of waves' shares and
of the launch shapes, both precisions, both stop rules, both spline ends,
with and without kept records."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one tile and less, tile edges, four waves of one tile, 16 waves of one tile
# (4096), the largest LDS-resident lengths (FP64 4660, FP32 8800), two to
# eight tiles per wave, and the longest the stage kernel takes (32768)
LENGTHS = [[4, 5, 63], [64, 65, 255, 256], [257, 511, 1000, 1024], [1025, 3000, 4096],
           [4097, 4600, 4700], [8192, 8600, 9100], [10007, 700], [16384, 16383], [30504],
           [32768, 5]]


def _inputs(dtype, lens):
    import torch
    sig = importlib.import_module("ceemdan-gpu_amd.signals")
    out = []
    for c, n in enumerate(lens):
        x = sig.eeg_like(n, seed=400 + c) if n >= 64 else np.random.default_rng(n).standard_normal(n)
        out.append(torch.tensor(x, dtype=dtype, device="cuda"))
    return out


def _steps(icm, plan):
    """Makes the plan take the launch-per-step path (default geometry)."""
    for ph in (icm.PHASE_NOISE, icm.PHASE_SIGNAL):
        plan.set_tuning(ph, [-1] * (plan.num_imfs - 1))


@pytest.mark.parametrize("lens", LENGTHS, ids=lambda v: "-".join(map(str, v)))
@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("stop,nak", [(0, 0), (0, 1), (1, 0)])
def test_stage_kernel_equals_steps(icm, dev, lens, dt, stop, nak):
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    I, M, S = 3, 4, 5
    print(f"case: whole stages {dt} stop={stop} nak={nak} lens={lens}", flush=True)
    xs = _inputs(dtype, lens)
    outs, modes = [], []
    for steps in (True, False):
        plan = icm.Plan(lens, I, M, dtype=dtype, stop_mode=stop, max_sifts=S, boundary=nak,
                        noise_max_sifts=S if stop == 0 else 70, use_graph=False, device=dev)
        if steps:
            _steps(icm, plan)
        outs.append([o.clone() for o in plan.forward(xs)])
        modes.append(plan.noise_modes())
        plan.close()
    for a, b in zip(*outs):
        assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
        assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(torch.nan_to_num(modes[0]), torch.nan_to_num(modes[1]))


@pytest.mark.parametrize("lens", [[300, 255, 4096], [9100, 700], [32768]],
                         ids=lambda v: "-".join(map(str, v)))
@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("keep", [True, False])
def test_stage_records_equal_steps(icm, dev, lens, dt, keep):
    """The knot structure that the stage kernel records gives the adjoint the
    same bits as the launch-per-step path's."""
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    I, M, S = 3, 4, 5
    print(f"case: stage records {dt} keep={keep} lens={lens}", flush=True)
    xs = _inputs(dtype, lens)
    rng = np.random.default_rng(3)
    gs = [torch.tensor(rng.standard_normal((M, n)), dtype=dtype, device="cuda") for n in lens]
    got = []
    for steps in (True, False):
        plan = icm.Plan(lens, I, M, dtype=dtype, max_sifts=S, use_graph=False, device=dev,
                        keep_records=keep)
        if steps:
            _steps(icm, plan)
        plan.forward(xs)
        got.append([g.clone() for g in plan.backward(gs)])
        plan.close()
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("rows,n", [(3, 4), (2, 256), (700, 257), (5, 4096), (3, 4600), (3, 4700),
                                    (2, 8600), (2, 9000), (2, 32768), (1, 70001)])
def test_sift_pass_routes(icm, orc, dev, dt, rows, n):
    """One pass, through one workgroup per series where its knots fit LDS and
    through the launch-per-step kernels where not: knot counts and samples of
    the oracle (FP64 equal, FP32 within 16 rounding errors of the largest
    sample, on the same float32 input), the same in place, and the same from
    the allocation-free entry."""
    import ctypes as C

    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    print(f"case: sift pass {dt} {rows} x {n}", flush=True)
    rng = np.random.default_rng(n)
    h = torch.tensor(rng.standard_normal((rows, n)), dtype=dtype, device="cuda")
    hn, nk = icm.sift_pass(h)
    for i in range(0, rows, max(1, rows // 3)):
        x = h[i].double().cpu().numpy()
        ref, nmax, nmin, _, _ = orc.sift_pass(x)
        assert nk[i].tolist() == [nmax, nmin]
        got = hn[i].double().cpu().numpy()
        if dt == "f64":
            assert np.array_equal(got, ref), i
        else:
            assert np.max(np.abs(got - ref)) <= 16 * 2.0 ** -24 * max(np.max(np.abs(x)), np.max(np.abs(ref)))
    st = C.c_void_p(torch.cuda.current_stream(h.device).cuda_stream)
    inplace, k2 = h.clone(), torch.zeros_like(nk)
    assert icm.lib().icm_sift_pass(icm._dtype_code(dtype), C.c_void_p(inplace.data_ptr()), n, rows,
                                   C.c_void_p(inplace.data_ptr()), C.c_void_p(k2.data_ptr()), st) == 0
    assert torch.equal(inplace, hn) and torch.equal(k2, nk)
    if rows * n <= 1 << 21:
        a, b = icm.sift_pass_static(h)
        assert torch.equal(a, hn) and torch.equal(b, nk)
