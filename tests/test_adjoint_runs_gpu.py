"""The adjoint viscosity gradient where its wave layout changes: one to six runs of
quads side by side (layers 2 to 33), one and two chunks of layers, runs that cross
strips and diamonds, both types."""
import numpy as np
import pytest

import oracle_lib as O
from fields import consistent_random


@pytest.mark.gpu
@pytest.mark.parametrize("lat,layers", [(1, 2), (3, 8), (3, 10), (3, 13), (2, 21), (3, 32), (3, 33), (2, 64), (2, 70),
                                        (5, 2)])
@pytest.mark.parametrize("bc", [(0, 0), (1, 2), (2, 2)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_grad_runs(cuda, lat, layers, bc, dtype):
    import torch

    import terraneo_amd as tn

    radii = np.linspace(0.55, 1.0, layers + 1) ** 1.1
    m, om = tn.Mesh(lat, radii=radii), O.Mesh(lat, radii=radii)
    td = getattr(torch, dtype)
    rng = np.random.default_rng(5)
    kc = np.exp(rng.random(10 * (m.n - 1) ** 2 * layers)).astype(dtype).astype("float64")
    u = consistent_random(om, 3, 3).reshape(-1).astype(dtype).astype("float64")
    lam = consistent_random(om, 3, 4).reshape(-1).astype(dtype).astype("float64")
    ref = O.Eps(om, None, *bc, kc=kc).grad_log_cell_viscosity(u, lam)
    op = tn.Eps(m, None, *bc, eta_cell=torch.from_numpy(kc).to(cuda, td))
    g = torch.full((kc.size,), float("nan"), dtype=td, device=cuda)
    op.grad_log_cell_eta(torch.from_numpy(u).to(cuda, td), torch.from_numpy(lam).to(cuda, td), g)
    err = np.abs(g.double().cpu().numpy() - ref).max() / np.abs(ref).max()
    # FP32: some 100 roundings along a term's way, 2^-24 each, of either sign: 10 x 6e-8,
    # with a factor of 30 for the terms (products of differences of rounded
    # coordinates over cells of 1/32) against their sum
    assert err <= (1e-12 if dtype == "float64" else 2e-5), err
