"""The couplings A12 and A21 with one lane per element, at the sizes where they
can go wrong: partial 8 x 8 tiles in either direction, one to many chunks of a
layer (test_gpu_lane_layers.py has chunks of several), one element, Dirichlet
dofs inside the box, and a mesh far from the origin (the pressure basis' frame
cancels); A21 of the smaller ones takes 27 lanes per element.

Tolerance: 1e-12 relative to the oracle, the bar of every FP64 operator here."""
import threading

import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray
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


def test_products_from_two_threads(gpu):
    """One operator's MatMult and A12 hand sums on through buffers of the operator:
    from two threads each gives what it gives alone, to the bit."""
    m = (40, 32, 32)
    rng = np.random.default_rng(5)
    E = m[0] * m[1] * m[2]
    A = MatStokesMF(*m).setup(F.box_coords(*m), F.eta_loguniform(E, 0.5, 2.0, rng), F.dirichlet_all_faces(*m))
    x = [DeviceArray.from_host(rng.uniform(-1, 1, n)) for n in (3 * F.nnodes(*m), 4 * E)]
    mult = (A.mult, A.mult_a12)
    alone = [DeviceArray(3 * F.nnodes(*m)) for _ in mult]
    for f, v, y in zip(mult, x, alone):
        f(v, y)
    ys = [[DeviceArray(3 * F.nnodes(*m)) for _ in range(30)] for _ in mult]
    threads = [threading.Thread(target=lambda f, v, out: [f(v, y) for y in out], args=a) for a in zip(mult, x, ys)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for want, out in zip(alone, ys):
        w = want.download()
        assert all(np.array_equal(w, y.download()) for y in out)
    A.destroy()


@pytest.mark.parametrize("m", [(1, 1, 7), (1, 1, 5000), (2, 3, 300), (16, 17, 18), (19, 20, 17)])
def test_divergence_of_thin_and_small_boxes(gpu, m):
    """A21 with 27 lanes per element, and the first boxes past that.  The oracle
    takes a few layers at a time, moved to the origin (exact differences): with
    5,000 elements to the unit it loses 1e-11 to the distance itself."""
    rng = np.random.default_rng(14)
    coords = F.perturb_interior(F.box_coords(*m), *m, 0.1, rng) + 5.0
    bc = F.dirichlet_all_faces(*m)
    bc[rng.integers(0, bc.size, bc.size // 20)] = 1
    A = MatStokesMF(*m).setup(coords, np.ones(27 * m[0] * m[1] * m[2]), bc)
    u = rng.uniform(-1.0, 1.0, bc.size)
    slab, plane = 8, 3 * (2 * m[0] + 1) * (2 * m[1] + 1)
    ref = []
    for k in range(0, m[2], slab):
        n = min(slab, m[2] - k)
        part = slice(2 * k * plane, (2 * (k + n) + 1) * plane)
        x = coords[part].reshape(-1, 3)
        ref.append(O.a21_matmult(m[0], m[1], n, (x - x[0]).reshape(-1), bc[part], u[part]))
    assert rel_inf(A.a21_host(u), np.concatenate(ref)) <= 1e-12
    A.destroy()
