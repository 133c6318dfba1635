"""The apply's even split of node columns over blocks: meshes whose runs are a
single column, cross from one strip into the next, and carry levels over a
radial chunk (64 cells) on both sides of such a crossing.

Bars as for every parity test of the apply: FP64 1e-12, FP32 5e-5 of max |y|.
"""
import numpy as np
import pytest

import oracle_lib as O
from fields import consistent_random, smooth_eta


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(1, 3), (4, 3), (4, 66), (5, 9), (5, 70)])
@pytest.mark.parametrize("dtype,bar", [("float64", 1e-12), ("float32", 5e-5)])
@pytest.mark.parametrize("bc", [(2, 2), (2, 1)])
def test_runs_across_strips(cuda, lat, nr, dtype, bar, bc):
    import torch

    import terraneo_amd as tn

    radii = np.linspace(0.55, 1.0, nr)
    m, om = tn.Mesh(lat, radii=radii), O.Mesh(lat, radii=radii)
    eta = smooth_eta(om.coords, om.radii).reshape(-1)
    x = consistent_random(om, 3, 5).reshape(-1)
    ref = O.Eps(om, eta, *bc).apply(x)
    dt = getattr(torch, dtype)
    op = tn.Eps(m, torch.from_numpy(eta).to(cuda, dt), *bc)
    xd = torch.from_numpy(x).to(cuda, dt)
    yd = torch.full_like(xd, float("nan"))
    op.apply(xd, yd)
    err = np.abs(yd.double().cpu().numpy() - ref).max() / np.abs(ref).max()
    assert err <= bar, err
