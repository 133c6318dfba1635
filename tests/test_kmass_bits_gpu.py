"""The lumped k-weighted mass to the last bit, at ten nodes of a level-1 shell (edges of
diamonds and a pole among them).  It is the Schur diagonal of the solves, and the CG on a
hierarchy's coarsest level amplifies its last bits.  The values are those of the row sums
of the quadrature's 6x6 matrices, formed one matrix after the other."""
import numpy as np
import pytest

from fields_exact import shell_fields

PINS = [(0, "0x1.f9e5962394bedp-7"), (1, "0x1.075a70bbeea98p-4"), (2, "0x1.cce6e74affb7bp-5"),
        (13, "0x1.715b194ac4b74p-4"), (40, "0x1.787b2e8b1cd07p-5"), (100, "0x1.26144e1261e65p-4"),
        (137, "0x1.557d2c7e9d40ep-5"), (200, "0x1.3ab3d2846e9ffp-4"), (255, "0x1.ac460fe8cbce8p-7"),
        (269, "0x1.2e29db6253280p-4")]


@pytest.mark.gpu
def test_lumped_mass_bits(cuda):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    m = tn.Mesh(1, radii=np.linspace(0.55, 1.0, 3))
    k = torch.from_numpy(shell_fields(m, 0)[0]).to(cuda)
    d = api.kmass_lumped(m, k, torch.empty_like(k)).cpu().numpy()
    assert [(i, float(d[i]).hex()) for i, _ in PINS] == PINS
