"""The MatMult of a box without Dirichlet dofs (an empty mask), with every kernel
that can form it: no launch may have nothing to do.

Tolerances: FP64 1e-12 and FP32 1e-5 relative to the oracle, the bars of every
MatMult here."""
import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray
from ptatin3d_amd.operators import BatchA11, MatA11MF

from conftest import rel_inf

pytestmark = pytest.mark.gpu


# box, kernel variant, tiles per work-group, tiling (None: the operator's own)
KERNELS = {"coloured": ((7, 5, 6), 3, 1, None), "coloured, one element": ((1, 1, 1), 3, 1, None),
           "column": ((7, 5, 6), 0, 1, None), "tile, one tile": ((3, 4, 2), 0, 1, (3, 4, 2)),
           "tile": ((7, 5, 6), 0, 1, (3, 2, 4)), "two tiles a group": ((7, 5, 6), 0, 2, None),
           "pipelined": ((7, 5, 6), 1, 1, None), "stored geometry": ((7, 5, 6), 2, 1, None),
           "lane": ((34, 31, 30), 0, 1, None)}


@pytest.mark.parametrize("kernel", list(KERNELS))
def test_matmult_without_dirichlet_dofs(gpu, kernel):
    m, variant, group, tiling = KERNELS[kernel]
    rng = np.random.default_rng(31)
    coords = F.box_coords(*m)
    if kernel != "lane":
        coords = F.perturb_interior(coords, *m, 0.1, rng)
    eta = F.eta_loguniform(m[0] * m[1] * m[2], 1e-2, 1e2, rng)
    bc = np.zeros(3 * F.nnodes(*m), np.uint8)
    u = rng.uniform(-1.0, 1.0, bc.size)
    A = MatA11MF(*m).setup(coords, eta, bc)
    if tiling:
        A.set_tiling(*tiling)
    A.set_kernel_variant(variant)
    A.set_tiles_per_group(group)
    yo = O.a11_matmult(*m, coords, eta, bc, u)
    assert rel_inf(A.mult_host(u), yo) <= 1e-12
    assert rel_inf(A.mult_host(u, precision=32), yo) <= 1e-5
    if variant != 3 and group == 1:
        B, x, y = BatchA11([A]), DeviceArray.from_host(u), DeviceArray(u.size)
        B.mult([x], [y], 64)
        assert rel_inf(y.download(), yo) <= 1e-12
        B.destroy()
    A.destroy()
