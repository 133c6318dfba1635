"""Nodal test fields made of sums and products of the mesh's coordinates alone, one value
per node: the same bits on every machine, for results pinned to their last bit."""
import numpy as np


def shell_fields(mesh, a):
    """A positive viscosity and a temperature, [N] each; `a` shifts them."""
    P, r = mesh.lateral_coords().reshape(-1, 3), np.asarray(mesh.radii())
    x, y, z = (P[:, k:k + 1] * r[None, :] for k in range(3))
    eta = 0.5 + (x + 0.1 * a) ** 2 * 3.0 + (y - z) ** 2 * 2.0 + 0.4 * z
    T = (1.0 - r[None, :]) * 2.0 + 0.3 * x * y - 0.2 * z * (x + 0.05 * a)
    # a node's copies lie a rounding apart: the first one's value at all of them
    place = np.round(P * 2 ** 30).astype(np.int64)
    _, first, inverse = np.unique(place, axis=0, return_index=True, return_inverse=True)
    pick = first[inverse.reshape(-1)]
    return tuple(np.ascontiguousarray(v[pick]).reshape(-1) for v in (eta, T))
