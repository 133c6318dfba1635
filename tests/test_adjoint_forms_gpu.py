"""The adjoint viscosity gradient by march and by cells: against the oracle on either side of
the rule that chooses (cells per lane, layers a wave holds), one to four runs side by side,
one chunk and two; and few cells cost little -- a quarter of a shell's layers at most 0.6 of
its time, where the march's start-up made it 0.9.

Bars against the oracle: FP64 1e-12; FP32 some 100 roundings along a term's way, 2^-24 each,
of either sign: 10 x 6e-8, with a factor of 60 for the terms (products of differences of
rounded coordinates over cells of 1/64) against their sum: 4e-5."""
import time

import numpy as np
import pytest

import oracle_lib as O
from fields import consistent_random


@pytest.mark.gpu
@pytest.mark.parametrize("lat,layers", [(7, 8), (7, 12), (6, 12), (6, 13), (6, 21), (6, 32), (5, 64), (5, 69), (5, 80), (5, 99)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_forms_against_oracle(cuda, lat, layers, dtype):
    import torch

    import terraneo_amd as tn

    bc = (1, 2) if layers % 2 else (2, 2)
    radii = np.linspace(0.55, 1.0, layers + 1) ** 1.1
    m, om = tn.Mesh(lat, radii=radii), O.Mesh(lat, radii=radii)
    td = getattr(torch, dtype)
    rng = np.random.default_rng(layers)
    kc = np.exp(rng.random(10 * (m.n - 1) ** 2 * layers)).astype(dtype).astype("float64")
    u = consistent_random(om, 3, 3).reshape(-1).astype(dtype).astype("float64")
    lam = consistent_random(om, 3, 4).reshape(-1).astype(dtype).astype("float64")
    ref = O.Eps(om, None, *bc, kc=kc).grad_log_cell_viscosity(u, lam)
    op = tn.Eps(m, None, *bc, eta_cell=torch.from_numpy(kc).to(cuda, td))
    g = torch.full((kc.size,), float("nan"), dtype=td, device=cuda)
    op.grad_log_cell_eta(torch.from_numpy(u).to(cuda, td), torch.from_numpy(lam).to(cuda, td), g)
    err = np.abs(g.double().cpu().numpy() - ref).max() / np.abs(ref).max()
    assert err <= (1e-12 if dtype == "float64" else 4e-5), err


@pytest.mark.gpu
def test_cost_of_few_layers(cuda):
    import torch

    import terraneo_amd as tn

    best = []
    for nr in (3, 9):
        m = tn.Mesh(7, radii=np.linspace(0.55, 1.0, nr))
        kc = torch.ones(10 * (m.n - 1) ** 2 * (nr - 1), device=cuda, dtype=torch.float64)
        u, g = torch.ones(3 * m.N, device=cuda, dtype=torch.float64), torch.empty_like(kc)
        op = tn.Eps(m, None, 2, 2, eta_cell=kc)
        best.append(float("inf"))
        for _ in range(5):
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(50):
                op.grad_log_cell_eta(u, u, g)
            torch.cuda.synchronize()
            best[-1] = min(best[-1], time.perf_counter() - t)
    assert best[0] <= 0.6 * best[1], best
