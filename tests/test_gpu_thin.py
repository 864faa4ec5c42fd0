"""The A11 diagonal and A12 of boxes with few elements or a thin cross-section,
where 27 lanes take an element in place of one: one element, columns and slabs
(one, two, four and eight parity classes with elements), and a slab past them.

Tolerance: 1e-12 relative to the oracle, the FP64 bar of both.  The oracle takes a
few layers at a time, moved to the origin (exact differences): with thousands of
elements to the unit it loses more than that to the distance."""
import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd.operators import MatStokesMF

from conftest import rel_inf

pytestmark = pytest.mark.gpu

LAYERS = 8


def _by_slabs(m, coords, nodal, element, f):
    """f(box, coordinates, nodal array, element array) put together from slabs
    that overlap by an element layer."""
    plane, layer = 3 * (2 * m[0] + 1) * (2 * m[1] + 1), element.size // m[2]
    out = []
    for k in range(0, m[2], LAYERS):
        lo, top = max(k - 1, 0), min(k + LAYERS, m[2])
        hi = min(top + 1, m[2])
        part = slice(2 * lo * plane, (2 * hi + 1) * plane)
        x = coords[part].reshape(-1, 3)
        y = f((m[0], m[1], hi - lo), (x - x[0]).reshape(-1), nodal[part], element[lo * layer:hi * layer])
        out.append(y[2 * (k - lo) * plane:(2 * (top - lo) + (top == m[2])) * plane])
    return np.concatenate(out)


@pytest.mark.parametrize("m", [(1, 1, 1), (1, 1, 300), (1, 200, 1), (2, 2, 12000), (100, 1, 400), (256, 1, 40)])
def test_diagonal_and_gradient_of_thin_boxes(gpu, m):
    rng = np.random.default_rng(14)
    E = m[0] * m[1] * m[2]
    coords = F.perturb_interior(F.box_coords(*m), *m, 0.1, rng) + 5.0
    bc = F.dirichlet_all_faces(*m)
    bc[rng.integers(0, bc.size, bc.size // 2)] = 0
    eta, p = F.eta_loguniform(E, 1e-2, 1e2, rng).reshape(-1), rng.uniform(-1.0, 1.0, 4 * E)
    A = MatStokesMF(*m).setup(coords, eta, bc)
    d, y = A.diagonal_host(), A.a12_host(p)
    assert rel_inf(d, _by_slabs(m, coords, bc, eta, lambda b, x, c, e: O.a11_diagonal(*b, x, e, c))) <= 1e-12
    assert np.all(d[bc.astype(bool)] == 1.0) and not y[bc.astype(bool)].any()
    assert rel_inf(y, _by_slabs(m, coords, bc, p, lambda b, x, c, q: O.a12_matmult(*b, x, c, q))) <= 1e-12
    assert np.array_equal(d, A.diagonal_host()) and np.array_equal(y, A.a12_host(p))  # no atomics
    A.destroy()
