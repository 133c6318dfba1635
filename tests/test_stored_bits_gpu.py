"""The stored apply forms every sum in one order, whichever way its rule splits a quad
over waves: a mesh of 640 quads and 8 layers (a wave per wedge) and the same mesh with
61 layers more on top (a wave per quad and chunk) give the same bits on the node levels
whose cells they share."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("bc", [0, 1, 2])
@pytest.mark.parametrize("dtype,store", [("float64", "f64"), ("float64", "f32"), ("float32", "f32")])
def test_same_bits_either_side_of_the_rule(cuda, bc, dtype, store):
    import torch

    import terraneo_amd as tn

    dt, low = getattr(torch, dtype), 9
    radii = np.concatenate([np.linspace(0.55, 0.7, low), np.linspace(0.7, 1.0, 62)[1:]])
    g = torch.Generator(device=cuda)
    g.manual_seed(17)
    tall, out = None, []
    for nr in (len(radii), low):
        m = tn.Mesh(3, radii=radii[:nr])
        if tall is None:
            tall = [torch.rand(k, 10 * m.n * m.n, m.nr, generator=g, device=cuda, dtype=torch.float64) for k in (1, 3)]
        eta, x = (v[..., :nr].contiguous().view(-1).to(dt) for v in tall)
        op = tn.Eps(m, 1.0 + eta, bc, tn.TN_NEUMANN)
        op.set_stored_matrices(tn.TN_F64 if store == "f64" else tn.TN_F32)
        out.append(op.apply(x, torch.empty_like(x)).view(3, -1, nr)[..., : low - 1])
    assert torch.equal(out[0], out[1])
