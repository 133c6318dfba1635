"""B and B^T as column stencils at the sizes where their walk changes: few
coarse columns, runs that end inside a strip, one to three chunks of levels with
lanes over at the end, both types, Replace and Add without exchange."""
import numpy as np
import pytest

import oracle_lib as O
from fields import consistent_random, smooth_eta


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("lat,rad,bc", [(2, 2, (2, 1)), (2, 6, (2, 2)), (2, 7, (1, 2)), (3, 8, (2, 2)), (5, 2, (0, 2))])
def test_coupling_columns(cuda, lat, rad, bc, dtype):
    import torch

    import terraneo_amd as tn

    td = getattr(torch, dtype)
    # sums of up to 3 * 5 * 19 products of tabulated factors: some 300 roundings of
    # either sign (sqrt(300) * eps of the largest value), with a factor of 20 for the
    # size of the terms against their sum
    bar = {"float64": 1e-12, "float32": 20 * 17.3 * 6e-8}[dtype]
    mv, mp = tn.Mesh(lat, rad, 0.55, 1.0), tn.Mesh(lat - 1, rad - 1, 0.55, 1.0)
    ov, op = O.Mesh(lat, mv.nr, 0.55, 1.0), O.Mesh(lat - 1, mp.nr, 0.55, 1.0)
    eta = torch.from_numpy(smooth_eta(ov.coords, ov.radii).reshape(-1)).to(cuda, td)
    K = tn.Stokes(mv, mp, tn.Eps(mv, eta, *bc))
    u = consistent_random(ov, 3, 11).reshape(-1).astype(dtype).astype("float64")
    p = consistent_random(op, 1, 12).reshape(-1).astype(dtype).astype("float64")
    ref_b = O.div_apply(ov, op, u, *bc)
    pd = torch.full((mp.N,), float("nan"), dtype=td, device=cuda)
    K.div(torch.from_numpy(u).to(cuda, td), pd)
    assert np.abs(pd.double().cpu().numpy() - ref_b).max() <= bar * np.abs(ref_b).max()
    ref_g = O.grad_apply_add(ov, op, p, np.zeros(3 * ov.N), *bc)
    pin = torch.from_numpy(p).to(cuda, td)
    ud = torch.full((3 * mv.N,), float("nan"), dtype=td, device=cuda)
    K.grad(pin, ud)
    assert np.abs(ud.double().cpu().numpy() - ref_g).max() <= bar * np.abs(ref_g).max()
    # the part of each copy, stored and added
    part = torch.empty_like(ud)
    K.grad(pin, part, comm_mode=tn.TN_COMM_SKIP)
    base = torch.from_numpy(u).to(cuda, td)
    both = base.clone()
    K.grad(pin, both, apply_mode=tn.TN_ADD, comm_mode=tn.TN_COMM_SKIP)
    assert torch.equal(both, base + part)
