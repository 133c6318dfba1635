"""The coarsest-level CG in one workgroup: a two-grid cycle whose coarse problem it
solves to rounding, against the same cycle with the dense inverse of the coarse
operator.  Coarse meshes with fewer and more nodes than threads, several radial
counts, every boundary pair that has a symmetric positive definite operator.

Bars: FP64 both coarse solves are exact to cond x 1e-13 with cond below 1e4 here:
1e-8 of max |x|.  FP32 coarse CG stops at 1e-6 of the residual, error at most
cond x 1e-6: 1e-2 of the coarse correction, which is part of x: 1e-2.
"""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(2, 5), (2, 7), (2, 17), (3, 9), (3, 5)])
@pytest.mark.parametrize("bc", [(1, 1), (2, 1), (2, 2)])
@pytest.mark.parametrize("dtype,store", [("float64", "f64"), ("float64", "f32"), ("float32", "f32")])
@pytest.mark.parametrize("zero", [True, False])
def test_two_grid_against_dense(cuda, lat, nr, bc, dtype, store, zero):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    dt = getattr(torch, dtype)
    radii = np.linspace(0.55, 1.0, nr)
    f, c = tn.Mesh(lat, radii=radii), tn.Mesh(lat - 1, radii=radii[::2])
    g = torch.Generator(device=cuda)
    g.manual_seed(11)
    eta = (1.0 + torch.rand(f.N, generator=g, device=cuda, dtype=torch.float64)).to(dt)
    A = api.Eps(f, eta, *bc)
    C = api.Eps(c, torch.ones(c.N, device=cuda, dtype=dt), *bc)
    for op in (A, C):
        op.set_penalty_once(True)
    C.gca_from(A, tn.TN_F64 if store == "f64" else tn.TN_F32)
    b = torch.rand(3 * f.N, generator=g, device=cuda, dtype=torch.float64).to(dt)
    f.interface_sum(b, 3)
    out = []
    for solver in ("pcg", "dense"):
        opts = api.gmg_options(cheby_order=2, cheby_iterations=1, coarse_solver=solver, coarse_max_iterations=2000,
                               coarse_rtol=1e-13 if dtype == "float64" else 1e-6, num_cycles=1 if zero else 2)
        gmg = api.Gmg([C, A], opts)
        x = torch.zeros_like(b)
        gmg.solve(x, b)
        out.append(x.double())
    err = float((out[0] - out[1]).abs().max() / out[1].abs().max())
    assert err <= (1e-8 if dtype == "float64" else 1e-2), err
