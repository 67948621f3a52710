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
