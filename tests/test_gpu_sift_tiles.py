"""The launch-per-step sift at its tile geometries against whole stages in one
workgroup: the same bits, for every remainder of a lane's four samples, one
to three samples in the last tile, segments of several tiles and less (a knot on
a tile's last sample is known to the next tile only), both tables, dense and
smooth series, and plateaus of equal samples."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [[4, 7, 9, 255, 257], [258, 259, 260, 513, 1021], [1279, 1281, 2050, 4099]]


def _series(n, kind):
    sig = importlib.import_module("ceemdan-gpu_amd.signals")
    if kind == "eeg" and n >= 64:
        return sig.eeg_like(n, seed=n)
    x = np.random.default_rng(n).standard_normal(n)
    return np.round(x * 2) / 2 if kind == "steps" else x


@pytest.mark.parametrize("lens", LENGTHS, ids=lambda v: "-".join(map(str, v)))
@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["eeg", "noise", "steps"])
def test_sift_geometries(icm, dev, lens, dt, kind):
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    I, M = 3, 4
    print(f"case: sift tiles {dt} {kind} lens={lens}", flush=True)
    xs = [torch.tensor(_series(n, kind), dtype=dtype, device="cuda") for n in lens]
    got = []
    for code in (None, -1, 0, 1, 2, 3):   # whole stages, default, 4 and 8 tiles, full and small table
        plan = icm.Plan(lens, I, M, dtype=dtype, max_sifts=6, use_graph=False, device=dev)
        if code is not None:
            for ph in (icm.PHASE_NOISE, icm.PHASE_SIGNAL):
                plan.set_tuning(ph, [code] * (M - 1))
        got.append([o.clone() for o in plan.forward(xs)] + [plan.noise_modes()])
        plan.close()
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
            assert torch.equal(torch.isnan(a), torch.isnan(b))
