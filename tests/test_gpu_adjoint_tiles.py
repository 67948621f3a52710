"""The adjoint's tile step at tile edges against the FP64 oracle's gradient:
one sample to one less than a tile in the last tile, every remainder of a
lane's four samples, dense noise (several knots per lane) and a slow tone
(tiles without knots)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [64, 255, 256, 257, 258, 259, 511, 512, 513, 1022, 1279, 2049])
@pytest.mark.parametrize("kind", ["noise", "tone"])
def test_adjoint_tile_edges(icm, orc, dev, N, kind):
    """Same measure and limit as for longer series (summation orders differ
    from the oracle's): relative max error of dL/dx <= 1e-9."""
    import torch
    I, M, S = 3, 4, 3
    rng = np.random.default_rng(N)
    x = rng.standard_normal(N)
    if kind == "tone":
        x = np.sin(2 * np.pi * np.arange(N) / 700.0) + 1e-3 * x
    G = rng.standard_normal((M, N))
    print(f"case: adjoint tiles {kind} N={N}", flush=True)
    w = icm.noise(I, N, seed=7, dtype=torch.float64, device=dev)
    plan = icm.Plan([N], I, M, dtype=torch.float64, max_sifts=S, use_graph=False, device=dev)
    out = plan.forward([torch.tensor(x, device=dev)], noise=w)[0].cpu().numpy()
    gx = plan.backward([torch.tensor(G, device=dev)])[0].cpu().numpy()
    plan.close()
    ref_g, ref_imfs = orc.iceemdan_grad(x, w.cpu().numpy(), M, G, S=S)
    assert np.array_equal(out, ref_imfs)
    assert np.max(np.abs(gx - ref_g)) <= 1e-9 * np.max(np.abs(ref_g))


@pytest.mark.parametrize("lens", [[700, 1025], [33000]], ids=lambda v: "-".join(map(str, v)))
@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_replayed_records(icm, dev, lens, dt):
    """Gradients after replayed graphs that keep their records, on new inputs
    each time, with eager work and synchronizations between: the same bits as
    from a plan that neither replays nor keeps them."""
    import torch
    dtype = torch.float64 if dt == "f64" else torch.float32
    I, M = 3, 4
    rng = np.random.default_rng(5)
    print(f"case: replayed records {dt} lens={lens}", flush=True)
    plans = [icm.Plan(lens, I, M, dtype=dtype, max_sifts=4, use_graph=g, keep_records=g, device=dev)
             for g in (True, False)]
    for _ in range(4):
        xs = [torch.tensor(rng.standard_normal(n), dtype=dtype, device="cuda") for n in lens]
        gs = [torch.tensor(rng.standard_normal((M, n)), dtype=dtype, device="cuda") for n in lens]
        got = []
        for p in plans:
            p.forward(xs)
            got.append([g.clone() for g in p.backward(gs)])
            torch.cuda.synchronize()
        for a, b in zip(*got):
            assert torch.equal(a, b)
    for p in plans:
        p.close()
