"""Destroying an object waits for the work queued with it, and a solve has finished when it
returns: the caller may then free or overwrite the arrays that the work reads, whichever
stream it was queued on."""
import numpy as np
import pytest


def _mesh(lat=6, nr=65):
    import terraneo_amd as tn

    return tn.Mesh(lat, radii=np.linspace(0.55, 1.0, nr))


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["eps", "stokes", "fv", "gmg"])
def test_destroy_waits(cuda, what):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    m, h = _mesh(), _mesh(5, 33)
    f64 = dict(device=cuda, dtype=torch.float64)
    eta, x = torch.ones(m.N, **f64), torch.zeros(3 * m.N, **f64)
    y, p = torch.empty_like(x), torch.zeros(h.N, **f64)
    A = tn.Eps(m, eta, 1, 1)
    if what == "eps":
        obj, call = A, lambda s: obj.apply(x, y, stream=s)
    elif what == "stokes":
        obj, call = tn.Stokes(m, h, A), lambda s: obj.grad(p, y, stream=s)
    elif what == "fv":
        obj = api.FV(m)
        T = obj.empty()
        call = lambda s: obj.to_fe_rhs(T, y, stream=s)  # noqa: E731
    else:
        C = tn.Eps(h, torch.ones(h.N, **f64), 1, 1)
        obj = api.Gmg([C, A], api.gmg_options(coarse_max_iterations=1))
        call = lambda s: obj.solve(y, x, stream=s)  # noqa: E731
    y.zero_()
    call(None)
    del A
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(100):
        call(s)
    del obj, call
    assert s.query()


@pytest.mark.gpu
def test_solve_has_finished(cuda):
    import torch

    from terraneo_amd import problem

    pr = problem.StokesProblem(5, 5, 2, 0.55, 1.0, bc=(1, 1), device=cuda)
    pr.set_viscosity(eta=torch.ones(pr.vel.N, **pr.f64))
    bu, bp = torch.ones(3 * pr.vel.N, **pr.f64), torch.zeros(pr.pre.N, **pr.f64)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        for its in (1, 2, 3):
            pr.solve(bu, bp, method="minres", max_iterations=its)
            assert s.query()
