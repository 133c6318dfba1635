"""Galerkin matrices at the edges of their 64-cell tiles (cell counts that are
and are not multiples of 64, a single coarse layer per quad upwards), from a
matrix-free and from a stored fine operator, nodal and per-cell viscosity:
with the geometric bracket the coarse operator is R A P exactly.

Bars: FP64 1e-12 of max |y| (sums of a few hundred products); FP32 storage
rounds each entry once, 2^-24 relative, and a row holds at most 63 entries of
comparable size: 63 x 6e-8 ~ 4e-6, bar 1e-5.
"""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(3, 9), (2, 13), (3, 21), (4, 9)])
@pytest.mark.parametrize("cell", [False, True])
@pytest.mark.parametrize("f32", [False, True])
def test_galerkin_is_rap(cuda, lat, nr, cell, f32):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    radii = np.linspace(0.55, 1.0, nr) ** 1.2
    meshes = [tn.Mesh(lat, radii=radii)]
    for k in (1, 2):
        meshes.append(tn.Mesh(lat - k, radii=radii[:: 1 << k]))
    g = torch.Generator(device=cuda)
    g.manual_seed(7)
    f = meshes[0]
    if cell:
        eta_c = 1.0 + torch.rand(10 * (f.n - 1) ** 2 * (f.nr - 1), generator=g, device=cuda, dtype=torch.float64)
        A = api.Eps(f, None, eta_cell=eta_c)
    else:
        A = api.Eps(f, 1.0 + torch.rand(f.N, generator=g, device=cuda, dtype=torch.float64))
    for m in meshes[1:]:
        C = api.Eps(m, torch.ones(m.N, device=cuda, dtype=torch.float64))
        C.gca_from(A, tn.TN_F32 if f32 else tn.TN_F64, bracket="geometric")
        x = torch.rand(3 * m.N, generator=g, device=cuda, dtype=torch.float64)
        m.interface_sum(x, 3)
        xf = torch.zeros(3 * f.N, device=cuda, dtype=torch.float64)
        api.prolongate_add(m, f, x, xf)
        yf, ref, y = torch.empty_like(xf), torch.empty_like(x), torch.empty_like(x)
        A.apply(xf, yf)
        api.restrict(f, m, yf, ref)
        C.apply(x, y)
        err = float((y - ref).abs().max() / ref.abs().max())
        assert err <= (1e-5 if f32 else 1e-12), err
        A, f = C, m
