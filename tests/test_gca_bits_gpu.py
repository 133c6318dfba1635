"""Galerkin matrices to the last bit: sum over the eight fine wedges of P^T (A P), every
product with P's powers of two exact, each sum in the order of its index -- written out
in numpy over the fine operator's wedge matrices as the library returns them.  From a
matrix-free and from a stored fine operator, both radial brackets, FP64 and FP32 storage."""
import numpy as np
import pytest

# fine wedges of a coarse wedge: cell offsets, wedge
LIST = [[(0, 0, 0, 0), (1, 0, 0, 0), (0, 1, 0, 0), (0, 0, 1, 0), (1, 0, 1, 0), (0, 1, 1, 0), (0, 0, 0, 1), (0, 0, 1, 1)],
        [(1, 0, 0, 1), (0, 1, 0, 1), (1, 1, 0, 1), (1, 0, 1, 1), (0, 1, 1, 1), (1, 1, 1, 1), (1, 1, 0, 0), (1, 1, 1, 0)]]
OFF = [[(0, 0), (1, 0), (0, 1)], [(1, 1), (0, 1), (1, 0)]]


def weights(fine, own):
    """[6 fine dofs][6 coarse dofs]; own: a lateral midpoint on the top plane takes the cell's top nodes."""
    P = np.zeros((6, 6))
    for i in range(6):
        m = i % 3
        a, b, c = fine[0] + OFF[fine[3]][m][0], fine[1] + OFF[fine[3]][m][1], fine[2] + i // 3
        if a % 2 == 0 and b % 2 == 0:
            P[i, [i] if c % 2 == 0 else [m, m + 3]] = 1.0 if c % 2 == 0 else 0.5
            continue
        e = (0, 2) if a % 2 == 0 else (0, 1) if b % 2 == 0 else (1, 2)
        for k in e:
            if c == 1:
                P[i, k] = P[i, k + 3] = 0.25
            else:
                P[i, k + (3 if c == 2 and own else 0)] = 0.5
    return P


def product(A, P):
    out = np.zeros((A.shape[0], P.shape[1]))
    for k in range(A.shape[1]):
        out = out + A[:, k:k + 1] * P[k:k + 1, :]
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("bracket", ["reference", "geometric"])
@pytest.mark.parametrize("f32", [False, True])
def test_galerkin_sums(cuda, bracket, f32):
    import torch

    import terraneo_amd as tn
    from terraneo_amd import api

    radii = np.linspace(0.55, 1.0, 9) ** 1.1
    meshes = [tn.Mesh(3 - k, radii=radii[:: 1 << k]) for k in range(3)]
    g = torch.Generator(device=cuda)
    g.manual_seed(23)
    eta = torch.rand(meshes[0].N, generator=g, device=cuda, dtype=torch.float64)
    A = api.Eps(meshes[0], torch.exp(4.0 * eta))
    for m in meshes[1:]:
        C = api.Eps(m, torch.ones(m.N, device=cuda, dtype=torch.float64))
        C.gca_from(A, tn.TN_F32 if f32 else tn.TN_F64, bracket=bracket)
        for d, x, y in ((0, 0, 0), (6, m.n - 2, 0), (9, m.n - 2, m.n - 2)):
            for r in range(m.nr - 1):
                for w in (0, 1):
                    out = np.zeros((18, 18))
                    for f in LIST[w]:
                        P = weights(f, bracket == "geometric" or r == m.nr - 2)
                        M = np.asarray(A.local_matrix(d, 2 * x + f[0], 2 * y + f[1], 2 * r + f[2], f[3])).reshape(18, 18)
                        for q in range(3):
                            for p in range(q, 3):
                                blk = M[6 * q:6 * q + 6, 6 * p:6 * p + 6]
                                out[6 * q:6 * q + 6, 6 * p:6 * p + 6] += product(P.T, product(blk, P))
                    ref = out.astype(np.float32).astype(np.float64) if f32 else out
                    got = np.asarray(C.local_matrix(d, x, y, r, w)).reshape(18, 18)
                    up = np.triu_indices(18)
                    assert np.array_equal(got[up], ref[up]), (m.n, d, x, y, r, w, abs(got[up] - ref[up]).max())
        A = C
