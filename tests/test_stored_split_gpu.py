"""The stored apply on both sides of the rule that gives a quad's wedges a wave each
(1024 waves on 256 compute units): meshes of 160, 640 and 2560 quads, one and two
chunks of layers, against the matrix-free apply of the same operator.

Bars: FP64 storage 1e-12 of max |y| (sums of a few hundred products); FP32 storage
rounds each entry once, 2^-24 relative, and a row holds at most 63 entries of
comparable size: 63 x 6e-8 ~ 4e-6, bar 1e-5."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("lat,nr", [(2, 3), (2, 67), (3, 9), (4, 5)])
@pytest.mark.parametrize("bc", [(0, 0), (1, 2), (2, 2)])
@pytest.mark.parametrize("f32", [False, True])
def test_stored_apply_small_levels(cuda, lat, nr, bc, f32):
    import torch

    import terraneo_amd as tn

    m = tn.Mesh(lat, radii=np.linspace(0.55, 1.0, nr) ** 1.1)
    g = torch.Generator(device=cuda)
    g.manual_seed(3)
    eta = 1.0 + torch.rand(m.N, generator=g, device=cuda, dtype=torch.float64)
    m.interface_sum(eta, 1)
    x = torch.rand(3 * m.N, generator=g, device=cuda, dtype=torch.float64)
    m.interface_sum(x, 3)
    free, st = tn.Eps(m, eta, *bc), tn.Eps(m, eta, *bc)
    st.set_stored_matrices(tn.TN_F32 if f32 else tn.TN_F64)
    ref, y = torch.empty_like(x), torch.empty_like(x)
    for comm in (tn.TN_COMM_ADDITIVE, tn.TN_COMM_SKIP):
        for mode in (tn.TN_REPLACE, tn.TN_ADD):
            for op, out in ((free, ref), (st, y)):
                op.set_modes(mode, comm)
                out.copy_(0.1 * x)
                op.apply(x, out)
            err = float((y - ref).abs().max() / ref.abs().max())
            assert err <= (1e-5 if f32 else 1e-12), (mode, comm, err)
