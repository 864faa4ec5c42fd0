"""The smoother's steps with the MatMult's last pass: Chebyshev from a zero and a
nonzero guess on a level of each element kernel (lane, column, tile with chunks of
several layers, coloured), against the recurrence on whole MatMults.

Tolerances: FP64 1e-12; FP32 1e-4: each of the four products rounds at up to
2e-6 of the result's size here and the recurrence at most doubles it per step."""
import numpy as np
import pytest

from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray
from ptatin3d_amd.multigrid import GMG, default_options
from ptatin3d_amd.operators import MatA11MF

from conftest import rel_inf

pytestmark = pytest.mark.gpu

KERNELS = {"lane": ((40, 32, 32), None, 0), "column": ((12, 20, 8), None, 0), "tile": ((8, 12, 20), (3, 2, 3), 0),
           "coloured": ((8, 4, 12), None, 3)}


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("nonzero", [True, False])
@pytest.mark.parametrize("kernel", list(KERNELS))
def test_smoother_against_whole_matmults(gpu, kernel, nonzero, bits):
    m, tiling, variant = KERNELS[kernel]
    rng = np.random.default_rng(8)
    mg = GMG(*m, 2)
    mg.set_coordinates(F.box_coords(*m))
    mg.set_viscosity(1, F.eta_loguniform(m[0] * m[1] * m[2], 0.5, 2.0, rng))
    mg.coarsen_viscosity("qp-arithmetic")
    bc = F.dirichlet_all_faces(*m)
    mg.set_dirichlet_all_faces()
    mg.setup(default_options(smoother_precision=bits))
    mg.set_eigs(1, 0.6, 3.3)
    A = MatA11MF.borrow(mg.level_op_handle(1), *m)
    if tiling:
        A.set_tiling(*tiling)
    A.set_kernel_variant(variant)
    d = A.diagonal_host()
    b = rng.uniform(-1, 1, bc.size)
    x0 = rng.uniform(-1, 1, bc.size) if nonzero else np.zeros(bc.size)
    scale = 2.0 / 3.9
    mu = 1.0 / (1.0 - scale * 0.6)
    p, c = [x0, x0 + scale * (b - A.mult_host(x0)) / d], [1.0, mu]
    for _ in range(3):
        c.append(2.0 * mu * c[-1] - c[-2])
        om = 2.0 * mu * c[-2] / c[-1]
        p.append(om * scale * (b - A.mult_host(p[-1])) / d + (1.0 - om) * p[-2] + om * p[-1])
    dt = np.float64 if bits == 64 else np.float32
    db, dx = DeviceArray.from_host(b.astype(dt)), DeviceArray.from_host(x0.astype(dt))
    mg.smooth(1, db, dx, 3, nonzero)
    assert rel_inf(dx.download(), p[-1]) <= (1e-12 if bits == 64 else 1e-4)
    A.set_kernel_variant(0)
    mg.destroy()
