"""Lane kernels whose waves march through several element layers, with partial
8 x 8 tiles and a shorter last chunk: the plane slots in LDS change places from
layer to layer, and a plane's sums are carried from one layer to the next.

65 x 47 x 41 has 2,214 tiles of one layer, so that 1,024 waves take chunks of 3 and
a last one of 2; 20 x 17 x 900 has 8,100, chunks of 8 and a last one of 4: every
place that a slot can have.  (In FP32, two waves a SIMD: 63 x 60 x 61 has 3,904 and
chunks of 2, the last of 1.)

Tolerances: FP64 1e-12 and FP32 1e-5 relative to the oracle, as everywhere here."""
import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray
from ptatin3d_amd.operators import MatStokesMF

from conftest import rel_inf

pytestmark = pytest.mark.gpu

BOXES = [(65, 47, 41), (20, 17, 900)]


def _case(m, mesh, seed):
    assert -(-m[0] // 8) * -(-m[1] // 8) * m[2] > 1024 and (m[0] % 8 or m[1] % 8)
    rng = np.random.default_rng(seed)
    E = m[0] * m[1] * m[2]
    coords = F.box_coords(*m).reshape(-1, 3) * (np.array(m) / max(m[:2]))  # (elements of about one shape)
    coords = coords.reshape(-1)
    if mesh == "deformed":
        coords = coords + 0.05 / max(m[:2]) * rng.uniform(-1.0, 1.0, coords.size)
    bc = F.dirichlet_all_faces(*m)
    bc[rng.integers(0, bc.size, bc.size // 40)] = 1
    eta = F.eta_loguniform(E, 1e-2, 1e2, rng)
    A = MatStokesMF(*m).setup(coords, eta, bc)
    u, p = rng.uniform(-1.0, 1.0, bc.size), rng.uniform(-1.0, 1.0, 4 * E)
    return A, coords, eta, bc, u, p, rng


@pytest.mark.parametrize("m", BOXES)
def test_couplings_and_coefficients(gpu, m):
    A, coords, eta, bc, u, p, rng = _case(m, "deformed", 41)
    assert rel_inf(A.a12_host(p), O.a12_matmult(*m, coords, bc, p)) <= 1e-12
    assert rel_inf(A.a21_host(u), O.a21_matmult(*m, coords, bc, u)) <= 1e-12
    assert rel_inf(A.diagonal_host(), O.a11_diagonal(*m, coords, eta, bc)) <= 1e-12
    B = 10.0 ** rng.uniform(-2.0, 2.0, 27 * A.nel)
    du, dB, de = DeviceArray.from_host(u), DeviceArray.from_host(B), DeviceArray(B.size)
    A.powerlaw_viscosity(du, dB, 3.0, 1e-3, 1e3, de)
    assert rel_inf(de.download(), O.powerlaw_eta(*m, coords, u, B, 3.0, 1e-3, 1e3)) <= 1e-12
    A.destroy()


@pytest.mark.parametrize("m", BOXES)
def test_matmult_and_saddle_point(gpu, m):
    A, coords, eta, bc, u, p, _ = _case(m, "box", 42)
    yo = O.a11_matmult(*m, coords, eta, bc, u)
    assert rel_inf(A.mult_host(u), yo) <= 1e-12
    yu, yp = A.stokes_host(u, p)
    assert rel_inf(yu, yo + O.a12_matmult(*m, coords, bc, p)) <= 1e-12
    assert rel_inf(yp, O.a21_matmult(*m, coords, bc, u)) <= 1e-12
    A.destroy()


def test_matmult_fp32(gpu):
    m = (63, 60, 61)
    A, coords, eta, bc, u, _, _ = _case(m, "box", 43)
    assert rel_inf(A.mult_host(u, precision=32), O.a11_matmult(*m, coords, eta, bc, u)) <= 1e-5
    A.destroy()
