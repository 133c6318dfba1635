"""Blocks of freed objects are reused safely: an operator destroyed while its
apply is still queued on a side stream, its replacement (same sizes) built and
applied at once on another stream; both results equal those of operators that
own their memory alone."""
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(2, 5), (4, 17)])
def test_reuse_across_streams(cuda, lat, nr):
    import numpy as np
    import torch

    import terraneo_amd as tn

    m = tn.Mesh(lat, radii=np.linspace(0.55, 1.0, nr))
    g = torch.Generator(device=cuda)
    g.manual_seed(3)
    etas = [1.0 + torch.rand(m.N, generator=g, device=cuda, dtype=torch.float64) for _ in range(4)]
    x = torch.rand(3 * m.N, generator=g, device=cuda, dtype=torch.float64)

    def stored(eta, stream=None):
        op = tn.Eps(m, eta, tn.TN_FREESLIP, tn.TN_FREESLIP)
        op.set_stored_matrices(tn.TN_F64, stream=stream)
        return op

    alone, ref = [stored(e) for e in etas], []
    for op in alone:
        ref.append(op.apply(x, torch.empty_like(x)))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in etas]
    out = [torch.empty_like(x) for _ in etas]
    for e, s, y in zip(etas, streams, out):
        op = stored(e, s)
        for _ in range(20):
            op.apply(x, y, stream=s)
        del op  # its applies may still be queued
    torch.cuda.synchronize()
    for y, r in zip(out, ref):
        assert torch.equal(y, r)
