"""The diagonal of A11 and the power-law viscosity with one lane per element, at
the sizes where they can go wrong: partial 8 x 8 tiles in either direction, one
to many chunks of a layer (test_gpu_lane_layers.py has chunks of several), one
element, Dirichlet dofs inside the box, sheared elements (the diagonal's mixed
products are large) and velocities at rest; the power law of the smaller ones
takes 27 lanes per element.

Tolerance: 1e-12 relative to the oracle, the FP64 bar of both operators."""
import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray
from ptatin3d_amd.operators import MatA11MF

from conftest import rel_inf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [(1, 1, 1), (8, 1, 2), (9, 5, 4), (17, 9, 11), (8, 8, 70), (30, 28, 33)])
def test_diagonal_and_powerlaw_parity(gpu, m):
    rng = np.random.default_rng(4)
    E = m[0] * m[1] * m[2]
    coords = F.perturb_interior(F.box_coords(*m), *m, 0.1, rng).reshape(-1, 3)
    coords[:, 0] += 0.7 * coords[:, 1] - 0.4 * coords[:, 2]
    coords = coords.reshape(-1)
    bc = F.dirichlet_all_faces(*m)
    bc[rng.integers(0, bc.size, bc.size // 20)] = 1
    eta = F.eta_loguniform(E, 1e-2, 1e2, rng)
    A = MatA11MF(*m).setup(coords, eta, bc)
    d = A.diagonal_host()
    assert rel_inf(d, O.a11_diagonal(*m, coords, eta, bc)) <= 1e-12
    assert np.all(d[bc.astype(bool)] == 1.0)
    assert np.array_equal(d, A.diagonal_host())  # no atomics: repeats are bit-identical

    u, B = rng.uniform(-1.0, 1.0, (F.nnodes(*m), 3)), 10.0 ** rng.uniform(-2.0, 2.0, 27 * E)
    u[: u.shape[0] // 3] = 0.0  # at rest: the floor of the strain rate
    ref = O.powerlaw_eta(*m, coords, u.reshape(-1), B, 3.0, 1e-3, 1e3)
    du, dB, de = DeviceArray.from_host(u.reshape(-1)), DeviceArray.from_host(B), DeviceArray(27 * E)
    A.powerlaw_viscosity(du, dB, 3.0, 1e-3, 1e3, de)
    assert rel_inf(de.download(), ref) <= 1e-12
    A.powerlaw_viscosity(du, dB, 3.0, 1e-3, 1e3, dB)  # in place
    assert np.array_equal(dB.download(), de.download())
    A.destroy()


@pytest.mark.parametrize("m", [(1, 1, 1), (9, 7, 1), (8, 4, 2), (13, 5, 1), (11, 6, 9)])
@pytest.mark.parametrize("tiling", [None, (4, 3, 2)])
def test_viscosity_copies(gpu, m, tiling):
    """The copies of a viscosity given on the device (63, 64, 65 elements and
    others; partial tiles and chunks) are those of one given on the host: the
    MatMults are bit-identical."""
    rng = np.random.default_rng(6)
    eta = F.eta_loguniform(m[0] * m[1] * m[2], 1e-2, 1e2, rng)
    coords = F.perturb_interior(F.box_coords(*m), *m, 0.1, rng)
    u = rng.uniform(-1.0, 1.0, 3 * F.nnodes(*m))
    ops = [MatA11MF(*m).setup(coords, e, F.dirichlet_all_faces(*m)) for e in (eta, np.ones_like(eta))]
    for A in ops:
        if tiling:
            A.set_tiling(*tiling)
    ops[1].set_viscosity_device(DeviceArray.from_host(eta.reshape(-1)))
    for prec in (64, 32):
        assert np.array_equal(ops[0].mult_host(u, precision=prec), ops[1].mult_host(u, precision=prec))
    for A in ops:
        A.destroy()


@pytest.mark.parametrize("m", [(1, 1, 7), (2, 3, 300), (70, 1, 60), (1, 64, 65), (26, 25, 31), (30, 25, 31)])
def test_powerlaw_of_thin_and_small_boxes(gpu, m):
    """27 lanes per element where a lane per element would leave most of a wave
    idle, and the first boxes past that: against the oracle, in place too."""
    rng = np.random.default_rng(14)
    coords = F.perturb_interior(F.box_coords(*m), *m, 0.1, rng) + 5.0
    E = m[0] * m[1] * m[2]
    u, B = rng.uniform(-1.0, 1.0, 3 * F.nnodes(*m)), 10.0 ** rng.uniform(-2.0, 2.0, 27 * E)
    A = MatA11MF(*m).setup(coords, np.ones(27 * E), F.dirichlet_all_faces(*m))
    ref = O.powerlaw_eta(*m, coords, u, B, 2.5, 1e-3, 1e3)
    du, dB = DeviceArray.from_host(u), DeviceArray.from_host(B)
    A.powerlaw_viscosity(du, dB, 2.5, 1e-3, 1e3, dB)
    assert rel_inf(dB.download(), ref) <= 1e-12
    A.destroy()
