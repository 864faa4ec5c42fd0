"""Material-point projection with per-element sums at the sizes where it can go
wrong: runs of one element shorter and longer than a wave's 64 points, points
in element order and in none, fewer points than a wave, a last wave that is
not full, one element with nearly all points.

The reference is the definition (_SwarmUpdateGaussPropertiesLocalL2Projection
Q1_MPntPStokes, material_point_utils.c:604-705,842-890) in NumPy.  All terms
are positive, so a sum of n terms in any order is within n eps of another:
with at most 5,000 points a node 1e-12 relative holds to the nodal field, and
the convex interpolation keeps it."""
import numpy as np
import pytest

from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray
from ptatin3d_amd.operators import MatA11MF

pytestmark = pytest.mark.gpu

S = np.sqrt(0.6)


def _reference(m, elem, xi, val):
    A = np.zeros([2 * k + 1 for k in reversed(m)])
    B = np.zeros_like(A)
    ei, ej, ek = elem % m[0], elem // m[0] % m[1], elem // (m[0] * m[1])
    f = [np.stack([0.5 * (1 - xi[:, d]), 0.5 * (1 + xi[:, d])]) for d in range(3)]
    lattice = [(i, j, k) for k in range(3) for j in range(3) for i in range(3)]
    for i, j, k in lattice:
        w = np.ones(val.size) if (i | j | k) & 1 else f[0][i // 2] * f[1][j // 2] * f[2][k // 2]
        np.add.at(A, (2 * ek + k, 2 * ej + j, 2 * ei + i), w * val)
        np.add.at(B, (2 * ek + k, 2 * ej + j, 2 * ei + i), w)
    e = np.arange(m[0] * m[1] * m[2])
    ei, ej, ek = e % m[0], e // m[0] % m[1], e // (m[0] * m[1])
    nod = np.stack([(A / B)[2 * ek + k, 2 * ej + j, 2 * ei + i] for i, j, k in lattice])
    g = np.array([[0.5 * (1 + S), 0.0, 0.5 * (1 - S)], [0.5, 0.0, 0.5], [0.5 * (1 - S), 0.0, 0.5 * (1 + S)]])
    v = np.einsum("rk,qj,pi,kjie->rqpe", g, g, g, nod.reshape(3, 3, 3, -1)).reshape(27, -1)
    return np.clip(v, nod.min(axis=0), nod.max(axis=0)).T


@pytest.mark.parametrize("m,per,order", [((1, 1, 1), 1, "element"), ((9, 5, 4), 2, "element"),
                                         ((9, 5, 4), 3, "none"), ((3, 8, 11), 5, "element"),
                                         ((4, 3, 2), 27, "one")])
def test_point_projection(gpu, m, per, order):
    rng = np.random.default_rng(11)
    E = m[0] * m[1] * m[2]
    elem = np.repeat(np.arange(E), per ** 3 if order != "one" else per)
    if order == "none":
        elem = rng.permutation(elem)
    if order == "one":
        elem = np.concatenate([elem[:E * per // 2], np.full(4001, 5), elem[E * per // 2:]])
    xi, val = rng.uniform(-1.0, 1.0, (elem.size, 3)), 10.0 ** rng.uniform(-2.0, 2.0, elem.size)
    A = MatA11MF(*m)
    eta = DeviceArray(27 * E)
    pts = [DeviceArray.from_host(v) for v in (elem.astype(np.int64), xi.reshape(-1), val)]
    ref = _reference(m, elem, xi, val)
    for _ in range(2):  # the workspace is used again
        A.project_points(*pts, eta)
        assert np.abs(eta.download().reshape(E, 27) / ref - 1.0).max() <= 1e-12
    A.destroy()
