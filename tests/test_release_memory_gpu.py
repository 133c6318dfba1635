"""Device memory of destroyed objects that the library keeps goes back on request, while
other objects live and keep working."""
import numpy as np
import pytest


@pytest.mark.gpu
def test_release_cached_memory(cuda):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    m = tn.Mesh(5, radii=np.linspace(0.55, 1.0, 33))
    eta = torch.ones(m.N, device=cuda, dtype=torch.float64)
    x = torch.rand(3 * m.N, device=cuda, dtype=torch.float64)
    kept = tn.Eps(m, eta, 1, 1)
    ref = kept.apply(x, torch.empty_like(x))
    for _ in range(2):  # (the first round also pays the runtime's own memory for these kernels)
        op = None
        api.release_cached_memory()
        before = torch.cuda.mem_get_info()[0]
        op = tn.Eps(m, eta, 1, 1)
        op.set_stored_matrices(tn.TN_F64)
    used = before - torch.cuda.mem_get_info()[0]
    assert used > 500 << 20  # 327680 cells x 2 x 172 x 8 bytes
    del op
    api.release_cached_memory()
    assert before - torch.cuda.mem_get_info()[0] < 64 << 20
    assert torch.equal(kept.apply(x, torch.empty_like(x)), ref)
