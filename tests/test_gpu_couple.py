"""The couplings A12 and A21 with one lane per element, at the sizes where they
can go wrong: partial 8 x 8 tiles in either direction, one to many layers a
chunk and a shorter last one, one element, Dirichlet dofs inside the box, and
a mesh far from the origin (the pressure basis' frame cancels).

Tolerance: 1e-12 relative to the oracle, the bar of every FP64 operator here."""
import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd.operators import MatStokesMF

from conftest import rel_inf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [(1, 1, 1), (8, 1, 2), (9, 5, 4), (17, 9, 11), (8, 8, 70), (30, 28, 33)])
def test_couplings_parity(gpu, m):
    rng = np.random.default_rng(4)
    E = m[0] * m[1] * m[2]
    coords = F.perturb_interior(F.box_coords(*m), *m, 0.1, rng) + 5.0
    bc = F.dirichlet_all_faces(*m)
    bc[rng.integers(0, bc.size, bc.size // 20)] = 1
    A = MatStokesMF(*m).setup(coords, np.ones(27 * E), bc)
    p, u = rng.uniform(-1.0, 1.0, 4 * E), rng.uniform(-1.0, 1.0, 3 * F.nnodes(*m))
    y = A.a12_host(p)
    assert np.abs(y - O.a12_matmult(*m, coords, bc, p)).max() <= 1e-12 * np.abs(p).max()
    assert not y[bc.astype(bool)].any()
    assert rel_inf(A.a21_host(u), O.a21_matmult(*m, coords, bc, u)) <= 1e-12
    assert np.array_equal(y, A.a12_host(p))  # no atomics: repeats are bit-identical
    A.destroy()
