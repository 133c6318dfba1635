"""A V-cycle whose coarsest level the one-workgroup CG solves has no host wait: it can be
captured, and every replay gives the eager cycle's bits.  (The queued CG waits for its
residuals, so a capture of it fails: this also pins which meshes take the one-workgroup
solve.)"""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(1, 3), (1, 9), (2, 5)])
@pytest.mark.parametrize("bc", [(1, 1), (2, 2)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_captured_cycle(cuda, lat, nr, bc, dtype):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    dt = getattr(torch, dtype)
    radii = np.linspace(0.55, 1.0, 2 * nr - 1)
    f, c = tn.Mesh(lat + 1, radii=radii), tn.Mesh(lat, radii=radii[::2])
    A = api.Eps(f, torch.ones(f.N, device=cuda, dtype=dt), *bc)
    C = api.Eps(c, torch.ones(c.N, device=cuda, dtype=dt), *bc)
    C.gca_from(A, tn.TN_F64 if dtype == "float64" else tn.TN_F32)
    gmg = api.Gmg([C, A], api.gmg_options(coarse_max_iterations=100))
    g = torch.Generator(device=cuda)
    g.manual_seed(37)
    b = torch.rand(3 * f.N, generator=g, device=cuda, dtype=torch.float64).to(dt)
    x = torch.zeros_like(b)
    gmg.solve(x, b)  # buffers and eigenvalue estimates
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.zero_()
        gmg.solve(x, b)
    for k in range(3):
        b.mul_(1.0 + 0.5 * k)
        ref = torch.zeros_like(b)
        gmg.solve(ref, b)
        x.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, ref)
