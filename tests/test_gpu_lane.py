"""The lane kernel of the A11 MatMult (rectilinear meshes, one lane per
element) at the sizes where it can go wrong: partial 8 x 8 tiles in either
direction, chunks of several layers with a shorter last one, Dirichlet dofs
inside the box, and meshes that only just are or are not rectilinear.

Tolerances: FP64 1e-12 relative to the oracle, the bar of every FP64 MatMult
here.  FP32 1e-5, likewise; the lane kernel's own FP32 roundings (about 40
along any path to a node value, 6e-8 each) stay below a quarter of it."""
import numpy as np
import pytest

from oracle import oracle as O
from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray, call
from ptatin3d_amd.multigrid import GMG, default_options, stokes_solve_timed
from ptatin3d_amd.operators import MatA11MF, MatStokesMF

from conftest import rel_inf

pytestmark = pytest.mark.gpu


def _axes(m, rng):
    """A rectilinear mesh with uneven element sizes (mid nodes halfway)."""
    ax = []
    for n in m:
        h = rng.uniform(0.5, 1.5, n)
        v = np.concatenate([[0.0], np.cumsum(h)]) / h.sum()
        a = np.empty(2 * n + 1)
        a[::2] = v
        a[1::2] = 0.5 * (v[:-1] + v[1:])
        ax.append(a)
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return np.stack([x, y, z], axis=-1).reshape(-1)


def _case(m, seed, uneven=True):
    rng = np.random.default_rng(seed)
    coords = _axes(m, rng) if uneven else F.box_coords(*m)
    eta = F.eta_loguniform(m[0] * m[1] * m[2], 1e-2, 1e2, rng)
    bc = F.dirichlet_all_faces(*m)
    bc[rng.integers(0, bc.size, bc.size // 40)] = 1
    u = rng.uniform(-1.0, 1.0, 3 * F.nnodes(*m))
    return coords, eta, bc, u


# (box, precision): each is past the size where the lane kernel takes over
BOXES = [((41, 33, 17), 64), ((17, 40, 35), 64), ((9, 25, 120), 64), ((64, 64, 23), 64), ((100, 4, 60), 64),
         ((64, 47, 20), 32), ((64, 61, 40), 32)]


@pytest.mark.parametrize("m,prec", BOXES)
def test_lane_matmult_parity(gpu, m, prec):
    coords, eta, bc, u = _case(m, 3)
    A = MatA11MF(*m).setup(coords, eta, bc)
    y = A.mult_host(u, precision=prec)
    yo = O.a11_matmult(*m, coords, eta, bc, u)
    tol = 1e-12 if prec == 64 else 1e-5
    assert rel_inf(y, yo) <= tol
    # Dirichlet rows are y = x exactly, and repeats are bit-identical
    d = bc.astype(bool)
    assert np.array_equal(y[d], u.astype(y.dtype)[d])
    assert np.array_equal(y, A.mult_host(u, precision=prec))
    if prec == 64:  # the tile kernel on the same operator (two tiles per work-group)
        A.set_tiles_per_group(2)
        assert rel_inf(A.mult_host(u), yo) <= tol
    A.destroy()


@pytest.mark.parametrize("move", [0.0, 1e-9])
def test_rectilinear_to_rounding_only(gpu, move):
    """One inner node off by 1e-9 of the box makes the mesh a general one: the
    MatMult must follow the coordinates it was given, and again after new
    rectilinear coordinates."""
    m = (32, 28, 30)
    coords, eta, bc, u = _case(m, 5, uneven=False)
    c = coords.reshape(2 * m[2] + 1, 2 * m[1] + 1, 2 * m[0] + 1, 3).copy()
    c[7, 9, 11, 1] += move
    A = MatA11MF(*m).setup(c.reshape(-1), eta, bc)
    assert rel_inf(A.mult_host(u), O.a11_matmult(*m, c.reshape(-1), eta, bc, u)) <= 1e-12
    c2 = _axes(m, np.random.default_rng(6))
    A.set_coordinates(c2)
    assert rel_inf(A.mult_host(u), O.a11_matmult(*m, c2, eta, bc, u)) <= 1e-12
    A.destroy()


def test_lane_noalloc_and_infinite_values(gpu):
    """The allocation-free entry point runs the same kernel (bit-identical),
    and an infinite input reaches the nodes of its own elements only."""
    m = (33, 30, 29)
    coords, eta, bc, u = _case(m, 7)
    bc = F.dirichlet_all_faces(*m)
    A = MatA11MF(*m).setup(coords, eta, bc)
    X, Y = 2 * m[0] + 1, 2 * m[1] + 1
    i, j, k = 2 * m[0] - 1, 2 * m[1] - 1, 21  # centre of the last element of a row
    u[3 * (i + X * (j + Y * k))] = np.inf
    x, y1, y2 = DeviceArray.from_host(u), DeviceArray(u.size), DeviceArray(u.size)
    A.mult(x, y1)
    call("ptmf_a11_mult_noalloc", A.handle, x.ptr, y2.ptr)
    call("ptmf_op_synchronize", A.handle)
    a = y1.download()
    assert np.array_equal(a, y2.download(), equal_nan=True)
    bad = ~np.isfinite(a.reshape(2 * m[2] + 1, Y, X, 3)).all(axis=-1)
    near = np.zeros_like(bad)
    near[k - 1:k + 2, j - 1:j + 2, i - 1:i + 2] = True
    assert bad.any() and not (bad & ~near).any()
    A.destroy()


def test_lane_smoother_takes_dirichlet_rows_itself(gpu):
    """The smoother's MatMult leaves the Dirichlet rows as element sums and its
    update takes y = x there: against the recurrence on whole MatMults, 1e-12."""
    m = (40, 32, 32)
    rng = np.random.default_rng(8)
    coords = F.box_coords(*m)
    mg = GMG(*m, 4)
    mg.set_coordinates(coords)
    mg.set_viscosity(3, F.eta_loguniform(m[0] * m[1] * m[2], 0.5, 2.0, rng))
    mg.coarsen_viscosity("qp-arithmetic")
    mg.set_dirichlet_all_faces()
    mg.setup(default_options(smoother_precision=64))
    mg.set_eigs(3, 0.6, 3.3)
    n = 3 * F.nnodes(*m)
    A = MatA11MF.borrow(mg.level_op_handle(3), *m)
    d = A.diagonal_host()
    b, x0 = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    scale = 2.0 / 3.9
    mu = 1.0 / (1.0 - scale * 0.6)
    p, c = [x0, x0 + scale * (b - A.mult_host(x0)) / d], [1.0, mu]
    for _ in range(3):
        c.append(2.0 * mu * c[-1] - c[-2])
        om = 2.0 * mu * c[-2] / c[-1]
        p.append(om * scale * (b - A.mult_host(p[-1])) / d + (1.0 - om) * p[-2] + om * p[-1])
    db, dx = DeviceArray.from_host(b), DeviceArray.from_host(x0)
    mg.smooth(3, db, dx, 3, True)
    assert rel_inf(dx.download(), p[-1]) <= 1e-12
    mg.destroy()


@pytest.mark.parametrize("m", [b for b, prec in BOXES if prec == 64])
def test_lane_saddle_point_parity(gpu, m):
    """MatMult_MFStokes_A with one lane per element = oracle A11 + A12 and A21."""
    coords, eta, bc, u = _case(m, 9)
    p = np.random.default_rng(10).uniform(-1.0, 1.0, 4 * m[0] * m[1] * m[2])
    A = MatStokesMF(*m).setup(coords, eta, bc)
    yu, yp = A.stokes_host(u, p)
    ou = O.a11_matmult(*m, coords, eta, bc, u) + O.a12_matmult(*m, coords, bc, p)
    op = O.a21_matmult(*m, coords, bc, u)
    assert rel_inf(yu, ou) <= 1e-12
    assert rel_inf(yp, op) <= 1e-12
    d = bc.astype(bool)
    assert np.array_equal(yu[d], u[d])
    A.set_tiles_per_group(2)  # the tile kernel on the same operator
    yu, yp = A.stokes_host(u, p)
    assert rel_inf(yu, ou) <= 1e-12
    assert rel_inf(yp, op) <= 1e-12
    A.destroy()


def test_lane_saddle_point_in_fp32_preconditioner(gpu):
    """The FP32 velocity preconditioner forms its A12 product with the FP32
    saddle-point kernel.  Its rounding, 1e-5 of the product, cannot show in a
    Krylov method's iterations to 1e-6 but for one at either end; a wrong
    product does."""
    m = (40, 32, 32)
    rng = np.random.default_rng(12)
    coords = F.box_coords(*m)
    eta = F.eta_loguniform(m[0] * m[1] * m[2], 0.1, 10.0, rng)
    its = []
    for prec in (64, 32):
        mg = GMG(*m, 3)
        mg.set_coordinates(coords)
        mg.set_viscosity(2, eta)
        mg.coarsen_viscosity()
        mg.set_dirichlet_all_faces()
        mg.setup(default_options(smoother_precision=prec))
        mg.stokes_setup()
        bu, bp = F.smooth_body_force(coords, *m), np.zeros(4 * m[0] * m[1] * m[2])
        out = stokes_solve_timed(mg, bu, bp, rtol=1e-6, maxit=200, restart=60)
        assert out[3] <= 1e-6 * np.linalg.norm(bu) * 1.5
        its.append(out[2])
        mg.destroy()
    assert abs(its[0] - its[1]) <= 1, its


@pytest.mark.parametrize("m", [(64, 47, 20), (31, 33, 64)])
def test_lane_fp32_in_si_units(gpu, m):
    """Elements of 100 km x 90 km x 10 km, viscosities about 1e25 Pa s and
    velocities about 1e-9 m/s: eta h^3 is past the largest FP32 number, every
    term of the result far from it."""
    coords, eta, bc, u = _case(m, 17)
    coords = (coords.reshape(-1, 3) * np.array([1e5, 9e4, 1e4]) * m).reshape(-1)
    eta, u = 1e25 * eta, 1e-9 * u
    A = MatA11MF(*m).setup(coords, eta, bc)
    y = A.mult_host(u, precision=32)
    assert np.isfinite(y).all()
    assert rel_inf(y, O.a11_matmult(*m, coords, eta, bc, u)) <= 1e-5
    A.destroy()


def test_kind_of_mesh_and_default_tiling(gpu):
    m = (12, 10, 9)
    coords, eta, bc, _ = _case(m, 19)
    A = MatA11MF(*m)
    default = A.get_tiling()
    assert not A.rectilinear
    A.setup(coords, eta, bc)
    assert A.rectilinear
    A.set_tiling(2, 2, 2)
    assert A.default_tiling() == default != A.get_tiling()
    A.set_coordinates(F.perturb_interior(coords, *m, 0.1, np.random.default_rng(1)))
    assert not A.rectilinear
    A.destroy()


def test_the_kernel_is_told(gpu):
    """Boxes on either side of the choices between tile, lane and column kernel,
    and each setting of the caller's."""
    for m, mesh, prec, want in (((28, 28, 28), "box", 64, "lane"), ((27, 27, 27), "box", 64, "column"),
                                ((30, 30, 30), "general", 64, "column"), ((48, 48, 48), "general", 64, "tile"),
                                ((48, 48, 48), "box", 32, "lane"), ((65, 40, 48), "box", 32, "tile")):
        A = MatA11MF(*m)
        x = F.box_coords(*m)
        A.set_coordinates(x if mesh == "box" else F.perturb_interior(x, *m, 0.1, np.random.default_rng(2)))
        assert A.mult_kernel(prec) == want, (m, mesh, prec)
        for v, name in ((1, "pipelined"), (2, "stored"), (3, "coloured")):
            A.set_kernel_variant(v)
            assert A.mult_kernel(prec) == name
        A.set_kernel_variant(0)
        A.set_tiles_per_group(2)
        assert A.mult_kernel(prec) == "tile"
        A.destroy()
