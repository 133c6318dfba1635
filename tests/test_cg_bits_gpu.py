"""Conjugate gradients without a preconditioner to the last bit: the solver's queued form
(scalars on the device) against the recurrence written out with the library's own vector
operations and a host scalar per reduction.  Meshes whose reductions have fewer blocks than
their cap and more, matrix-free and stored operators, iteration counts within and past a
batch, and a tolerance that ends the solve."""
import numpy as np
import pytest


def recurrence(m, A, x, b, cap, rtol=0.0):
    """The iterates and residuals of a solve from x; x is replaced."""
    import torch

    r, ap = torch.empty_like(b), torch.empty_like(b)
    A.apply(x, r)
    m.lincomb(r, [1.0, -1.0], [b, r])
    p, rr = r.clone(), m.dot(r, r, 3)
    hist = [np.sqrt(rr)]
    for _ in range(cap):
        A.apply(p, ap)
        a = rr / m.dot(ap, p, 3)
        m.lincomb(x, [1.0, a], [x, p])
        m.lincomb(r, [1.0, -a], [r, ap])
        new = m.dot(r, r, 3)
        hist.append(np.sqrt(new))
        if hist[-1] / hist[0] <= rtol:
            break
        m.lincomb(p, [1.0, new / rr], [r, p])
        rr = new
    return hist


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr,bc", [(2, 5, (2, 2)), (3, 67, (1, 2)), (5, 33, (1, 1)), (6, 9, (2, 2))])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("stored", [False, True])
def test_queued_is_the_recurrence(cuda, lat, nr, bc, dtype, stored):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    dt = getattr(torch, dtype)
    m = tn.Mesh(lat, radii=np.linspace(0.55, 1.0, nr) ** 1.1)
    g = torch.Generator(device=cuda)
    g.manual_seed(5)
    eta = 1.0 + torch.rand(m.N, generator=g, device=cuda, dtype=torch.float64)
    m.interface_sum(eta, 1)
    A = tn.Eps(m, eta.to(dt), *bc)
    if stored:
        A.set_stored_matrices(tn.TN_F64 if dtype == "float64" else tn.TN_F32)
    b = torch.rand(3 * m.N, generator=g, device=cuda, dtype=torch.float64).to(dt)
    m.interface_sum(b, 3)
    x0 = torch.rand(3 * m.N, generator=g, device=cuda, dtype=torch.float64).to(dt)
    m.interface_sum(x0, 3)
    for cap, rtol in ((1, 0.0), (7, 0.0), (27, 0.0), (60, 0.2)):
        ref, x = x0.clone(), x0.clone()
        hist = recurrence(m, A, ref, b, cap, rtol)
        info = api.pcg_solve(A, x, b, max_iterations=cap, rtol=rtol, atol=0.0)
        assert info["history"].tolist() == hist
        assert torch.equal(x, ref)
