"""The stable step and the FCT predictor by columns and by cells: against the oracle on
either side of the rule that chooses (layers a chunk of 64 lanes holds, columns a CU gets),
one chunk and two, and a shell of few layers at about the thick shell's cost per cell.

Bars against the oracle: 1e-12 relative (max norm), some 1e3 roundings of FP64 terms no
larger than 4 times their sum.  Cost: twice per cell, where lanes empty but for 8 layers
of 64 made it four times."""
import time

import numpy as np
import pytest

import fv_oracle_lib as F
import oracle_lib as O


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(5, 24), (5, 27), (5, 40), (5, 42), (5, 68), (5, 83), (4, 83)])
def test_forms_against_oracle(cuda, lat, nr):
    import torch

    from terraneo_amd import api

    radii = 0.55 + 0.45 * np.linspace(0.0, 1.0, nr) ** 1.3
    gm, om = api.Mesh(lat, radii=radii), O.Mesh(lat, radii=radii)
    fv, co = api.FV(gm), F.cell_centers(om)
    rng = np.random.default_rng(nr)
    X = om.node_xyz()
    rot = np.cross(np.array([0.5, -0.3, 0.8])[None, None, None, None, :], X)
    vel = np.ascontiguousarray(np.moveaxis(rot, -1, 0) + 0.2 * rng.uniform(-1, 1, (3,) + om.shape)).reshape(-1)
    T = rng.uniform(0, 1, F.fv_shape(om))
    vg, Tg = torch.from_numpy(vel).to(cuda), torch.from_numpy(T).to(cuda)
    dt, dto = fv.dt_stable(vg, 0.03), F.dt_stable(om, co, vel, 0.03)
    assert abs(dt - dto) <= 1e-12 * dto
    fv.predictor(Tg, vg, 0.5 * dto, 0.03)
    TL, ad, _, _ = fv.buffers()
    _, TLo, ado = F.predictor(om, co, vel, T, 0.5 * dto, 0.03)
    real = (Ellipsis,) + (slice(1, -1),) * 3
    assert np.abs(TL[real] - TLo[real]).max() <= 1e-12 * np.abs(TLo[real]).max()
    ado = np.moveaxis(ado, -1, 0)
    assert np.abs(ad[real] - ado[real]).max() <= 1e-12 * np.abs(ado[real]).max()


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["dt", "predictor"])
def test_cost_of_a_thin_shell(cuda, what):
    import torch

    from terraneo_amd import api

    cost = []
    for nr in (9, 41):
        m = api.Mesh(7, radii=np.linspace(0.55, 1.0, nr))
        fv = api.FV(m)
        T = torch.zeros(fv.fv_shape, device=cuda, dtype=torch.float64)
        u = torch.ones(3 * m.N, device=cuda, dtype=torch.float64)
        best = float("inf")
        for _ in range(5):
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(10):
                fv.dt_stable(u, 1.0) if what == "dt" else fv.predictor(T, u, 1e-7, 1.0)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        cost.append(best / (nr - 1))
    # (the stable step's call also costs a host round trip of 25 us whatever the mesh)
    assert cost[0] <= (3.5 if what == "dt" else 2.0) * cost[1], cost
