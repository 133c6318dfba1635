"""Restriction as the transpose of the prolongation over owned nodes, both types, one
and three components, on the smallest meshes and past 64 levels."""
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("lat,rad", [(1, 2), (2, 2), (3, 7), (4, 3)])
@pytest.mark.parametrize("ncomp", [1, 3])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_restrict_is_transpose(cuda, lat, rad, ncomp, dtype):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    td = getattr(torch, dtype)
    f, c = tn.Mesh(lat, rad, 0.55, 1.0), tn.Mesh(lat - 1, rad - 1, 0.55, 1.0)
    g = torch.Generator(device=cuda)
    g.manual_seed(1)
    xf = torch.rand(ncomp * f.N, generator=g, device=cuda, dtype=td) - 0.5
    f.interface_sum(xf, ncomp)
    xc = torch.rand(ncomp * c.N, generator=g, device=cuda, dtype=td) - 0.5
    c.interface_sum(xc, ncomp)
    rf = torch.full_like(xc, float("nan"))
    api.restrict(f, c, xf, rf, ncomp=ncomp)
    pc = torch.zeros_like(xf)
    api.prolongate_add(c, f, xc, pc, ncomp=ncomp)
    a, b = c.dot(rf, xc, ncomp), f.dot(xf, pc, ncomp)
    # each product rounds some 40 times on its way, 2^-53 or 2^-24 each, of either sign,
    # relative to |x| |y|
    scale = (c.dot(rf, rf, ncomp) * c.dot(xc, xc, ncomp)) ** 0.5
    assert abs(a - b) <= (1e-14 if dtype == "float64" else 4e-6) * scale, (a, b, scale)
