"""Conjugate gradients with their scalars on the device, against the recurrence
written out with the library's host-side vector operations: iteration counts that
end inside, at the end of and after a batch of eight, the iteration cap, and
meshes with one radial column chunk, a remainder and two.

Both sides run the same FP64 recurrence; their sums differ in order, so the
residuals agree to the conditioning of a short solve: 1e-9 of the first one.
"""
import numpy as np
import pytest


def _reference(m, A, x, b, its, ncomp):
    import torch

    r, ap = torch.empty_like(b), torch.empty_like(b)
    A(x, r)
    r = b - r
    p, rr = r.clone(), m.dot(r, r, ncomp)
    hist = [np.sqrt(rr)]
    for _ in range(its):
        A(p, ap)
        a = rr / m.dot(ap, p, ncomp)
        x = x + a * p
        r = r - a * ap
        new = m.dot(r, r, ncomp)
        p, rr = r + new / rr * p, new
        hist.append(np.sqrt(rr))
    return x, np.array(hist)


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(1, 3), (2, 5), (3, 64), (3, 65), (4, 17)])
@pytest.mark.parametrize("its", [1, 7, 8, 9, 16, 21])
def test_projection_cg(cuda, lat, nr, its):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    m = tn.Mesh(lat, radii=np.linspace(0.55, 1.0, nr))
    fv = api.FV(m)
    g = torch.Generator(device=cuda)
    g.manual_seed(its)
    T = torch.rand(fv.fv_shape, generator=g, device=cuda, dtype=torch.float64)
    x0 = torch.rand(m.N, generator=g, device=cuda, dtype=torch.float64)
    m.interface_sum(x0, 1)
    b = torch.empty_like(x0)
    fv.to_fe_rhs(T, b)
    one = torch.ones_like(b)

    def mass(v, y):  # component 0 of the vector mass
        z = torch.zeros(3 * m.N, device=cuda, dtype=torch.float64)
        z[: m.N] = v
        o = torch.empty_like(z)
        api.vector_mass(m, z, o)
        y.copy_(o[: m.N])

    ref, hist = _reference(m, mass, x0.clone(), b, its, 1)
    x = x0.clone()
    info = fv.to_fe(T, x, max_iterations=its, rtol=0.0, atol=0.0)
    assert info["iterations"] == its and len(info["history"]) == its + 1
    assert np.abs(info["history"] - hist).max() <= 1e-9 * hist[0]
    assert float((x - ref).abs().max()) <= 1e-9 * float(ref.abs().max())
    # a tolerance met at iteration k stops there, whatever is queued behind
    k = max(1, its - 1)
    tol = np.sqrt(hist[k] * hist[k - 1]) / hist[0]  # between the two residuals
    if hist[: k].min() / hist[0] > tol:
        y = x0.clone()
        i2 = fv.to_fe(T, y, max_iterations=its + 20, rtol=tol, atol=0.0)
        assert i2["iterations"] == k


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_operator_cg(cuda, dtype):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    dt = getattr(torch, dtype)
    m = tn.Mesh(3, 3, 0.55, 1.0)
    A = tn.Eps(m, torch.ones(m.N, device=cuda, dtype=dt), tn.TN_DIRICHLET, tn.TN_DIRICHLET)
    g = torch.Generator(device=cuda)
    g.manual_seed(1)
    b = torch.rand(3 * m.N, generator=g, device=cuda, dtype=torch.float64).to(dt)
    m.interface_sum(b, 3)
    ref, hist = _reference(m, lambda v, y: A.apply(v, y), torch.zeros_like(b), b, 12, 3)
    x = torch.zeros_like(b)
    info = api.pcg_solve(A, x, b, max_iterations=12, rtol=0.0, atol=0.0)
    bar = 1e-9 if dtype == "float64" else 1e-3  # 12 steps of 2^-24 rounding, growth below 1e3
    assert np.abs(info["history"] - hist).max() <= bar * hist[0]
    assert float((x - ref).abs().max()) <= bar * float(ref.abs().max())
