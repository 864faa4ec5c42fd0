"""The column kernel of the A11 MatMult (small boxes, one lane per node column) at
the sizes where it can go wrong: fewer elements than a wave's five, a last wave
that is not full, one element in a direction, the largest box it takes (103,563
elements) and one past it, Dirichlet dofs inside the box, alone and in a batch.

Tolerances: FP64 1e-12 relative to the oracle, FP32 5e-5, the bars of every
MatMult here."""
import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray, call
from ptatin3d_amd.operators import BatchA11, MatA11MF

from conftest import rel_inf

pytestmark = pytest.mark.gpu


def _case(m, seed, perturbed=True):
    rng = np.random.default_rng(seed)
    coords = F.box_coords(*m)
    if perturbed:
        coords = F.perturb_interior(coords, *m, 0.1, rng) + 2.0
    eta = F.eta_loguniform(m[0] * m[1] * m[2], 1e-2, 1e2, rng)
    bc = F.dirichlet_all_faces(*m)
    bc[rng.integers(0, bc.size, max(1, bc.size // 40))] = 1
    return coords, eta, bc, rng.uniform(-1.0, 1.0, 3 * F.nnodes(*m))


@pytest.mark.parametrize("m,perturbed", [((1, 1, 1), True), ((2, 1, 2), True), ((5, 1, 1), True), ((1, 1, 11), True),
                                         ((13, 1, 7), True), ((16, 15, 17), True), ((12, 12, 12), False),
                                         ((47, 47, 46), True), ((47, 47, 47), True)])
def test_column_kernel_parity(gpu, m, perturbed):
    coords, eta, bc, u = _case(m, 3, perturbed)
    A = MatA11MF(*m).setup(coords, eta, bc)
    yo = O.a11_matmult(*m, coords, eta, bc, u)
    y = A.mult_host(u)
    assert rel_inf(y, yo) <= 1e-12
    if m != (47, 47, 47):  # there the tile kernel runs, whose FP32 rounding grows with the distance from the origin
        assert rel_inf(A.mult_host(u, precision=32), yo) <= 5e-5
    d = bc.astype(bool)
    assert np.array_equal(y[d], u[d])
    assert np.array_equal(y, A.mult_host(u))
    A.set_tiles_per_group(2)  # the tile kernel on the same operator
    assert rel_inf(A.mult_host(u), yo) <= 1e-12
    A.destroy()


def test_column_kernel_infinite_values(gpu):
    """An infinite input reaches the nodes of its own elements only."""
    m = (6, 5, 4)
    coords, eta, _, u = _case(m, 4)
    bc = F.dirichlet_all_faces(*m)
    A = MatA11MF(*m).setup(coords, eta, bc)
    X, Y, Z = (2 * k + 1 for k in m)
    i, j, k = 5, 3, 3  # the centre of an element
    u[3 * (i + X * (j + Y * k))] = np.inf
    x, y1, y2 = DeviceArray.from_host(u), DeviceArray(u.size), DeviceArray(u.size)
    A.mult(x, y1)
    call("ptmf_a11_mult_noalloc", A.handle, x.ptr, y2.ptr)
    call("ptmf_op_synchronize", A.handle)
    a = y1.download()
    assert np.array_equal(a, y2.download(), equal_nan=True)
    bad = ~np.isfinite(a.reshape(Z, Y, X, 3)).all(axis=-1)
    near = np.zeros_like(bad)
    near[k - 1:k + 2, j - 1:j + 2, i - 1:i + 2] = True
    assert bad.any() and not (bad & ~near).any()
    A.destroy()


def test_batch_of_both_kernels(gpu):
    """Boxes with a tiling of the caller's own among boxes of the column kernel,
    and again after one of them changes over."""
    boxes = [(4, 4, 4), (7, 3, 5), (1, 9, 2), (8, 8, 8)]
    cases = [_case(m, 20 + i) for i, m in enumerate(boxes)]
    ops = [MatA11MF(*m).setup(c, e, b) for m, (c, e, b, _) in zip(boxes, cases)]
    ops[1].set_tiling(3, 2, 2)
    batch = BatchA11(ops)
    refs = [O.a11_matmult(*m, c, e, b, u) for m, (c, e, b, u) in zip(boxes, cases)]
    for change in (None, 3, 0):
        if change is not None:
            ops[change].set_tiling(2, 2, 1)
        for prec, dt, tol in ((64, np.float64, 1e-12), (32, np.float32, 5e-5)):
            xs = [DeviceArray.from_host(c[3].astype(dt)) for c in cases]
            ys = [DeviceArray(c[3].size, dt) for c in cases]
            batch.mult(xs, ys, precision=prec)
            for y, ref in zip(ys, refs):
                assert rel_inf(y.download(), ref) <= tol
    batch.destroy()
    for A in ops:
        A.destroy()
