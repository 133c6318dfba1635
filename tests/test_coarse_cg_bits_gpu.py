"""The coarsest-level CG to the last bit: a two-level cycle without smoothing is restriction,
coarse solve and prolongation, so its even nodes are the coarse solution.  They equal the
recurrence written out with the library's vector operations: the default tolerance, a loose
one met mid-solve, small iteration caps, an absolute tolerance above the first residual.
Meshes for one copy per thread, for four and past the one-workgroup solve; every boundary pair,
the penalty at every copy and at the owned one."""
import numpy as np
import pytest

from test_cg_bits_gpu import recurrence


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(1, 3), (1, 9), (2, 5), (0, 17), (2, 9)])
@pytest.mark.parametrize("bc,once", [((0, 0), False), ((1, 1), False), ((2, 1), False), ((2, 2), False), ((2, 2), True)])
@pytest.mark.parametrize("dtype,store", [("float64", "f64"), ("float64", "f32"), ("float32", "f32")])
def test_coarse_solve_is_the_recurrence(cuda, lat, nr, bc, once, dtype, store):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    dt = getattr(torch, dtype)
    radii = np.linspace(0.55, 1.0, 2 * nr - 1) ** 1.1
    f, c = tn.Mesh(lat + 1, radii=radii), tn.Mesh(lat, radii=radii[::2])
    g = torch.Generator(device=cuda)
    g.manual_seed(29)
    eta = 1.0 + 9.0 * torch.rand(f.N, generator=g, device=cuda, dtype=torch.float64)
    f.interface_sum(eta, 1)
    A = api.Eps(f, eta.to(dt), *bc)
    C = api.Eps(c, torch.ones(c.N, device=cuda, dtype=dt), *bc)
    for op in (A, C):
        op.set_penalty_once(once)
    C.gca_from(A, tn.TN_F64 if store == "f64" else tn.TN_F32)
    b = torch.rand(3 * f.N, generator=g, device=cuda, dtype=torch.float64).to(dt)
    f.interface_sum(b, 3)
    bc_ = api.restrict(f, c, b, torch.empty(3 * c.N, device=cuda, dtype=dt))
    # (a pure Neumann operator is singular: short solves)
    for cap, rtol, atol in ((1, 1e-6, 1e-16), (7, 1e-6, 1e-16), (40 if bc == (0, 0) else 400, 1e-6, 1e-16),
                            (40, 0.1, 1e-16), (40, 1e-6, 1e30)):
        gmg = api.Gmg([C, A], api.gmg_options(cheby_iterations=0, coarse_max_iterations=cap, coarse_rtol=rtol,
                                              coarse_atol=atol))
        x = gmg.solve(torch.zeros_like(b), b)
        ref = torch.zeros_like(bc_)
        if float(np.sqrt(c.dot(bc_, bc_, 3))) >= atol:
            recurrence(c, C, ref, bc_, cap, rtol)
        got = x.view(3, 10, f.n, f.n, f.nr)[:, :, ::2, ::2, ::2]
        assert torch.equal(got, ref.view(3, 10, c.n, c.n, c.nr)), (cap, rtol, atol)
