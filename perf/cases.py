"""Workloads that the speed of the operator stack is measured on.

Each case is work that a program using this framework has it do, through its
public entry points: the viscous MatMult that every Krylov iteration and
smoothing step calls (in both precisions, from the latency-bound smallest box
to the largest), the fused saddle-point MatMult, the pressure couplings, the
coefficient update of a Picard step, the material-point projection, a
smoother call, a V-cycle and a batched MatMult.

  listed()            the cases
  draw(rng)           one more of the same ranges
  prepare(case, seed) what a program has in hand before the call
  run(state)          one pass, its outputs as tensors
  work(case)          the bytes and operations the pass cannot do without
  exact(case, seed)   the outputs in plain 64-bit torch, where that is quick
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from ptatin3d_amd import fields as F
from ptatin3d_amd._lib import DeviceArray, call
from ptatin3d_amd.multigrid import GMG, default_options
from ptatin3d_amd.operators import BatchA11, MatA11MF, MatStokesMF

# executed arithmetic of one element (the sum-factorised form; the reference
# counts 17,253 for its tensor kernel)
A11_FLOPS = 10800
MAX_ELEMENTS = 128 ** 3


class TensorArray(DeviceArray):
    """A tensor's memory as the framework's device array (the tensor owns it)."""

    _dtypes = {torch.float64: np.float64, torch.float32: np.float32, torch.int64: np.int64}

    def __init__(self, t: torch.Tensor):
        assert t.is_contiguous()
        self.tensor = t
        self.dtype = np.dtype(self._dtypes[t.dtype])
        self.n = t.numel()
        self.nbytes = self.n * self.dtype.itemsize
        self.ptr = C.c_void_p(t.data_ptr())

    def free(self) -> None:
        self.tensor = None
        self.ptr = None

    def __del__(self):
        pass


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # the MatMult of the smallest solves and of the coarse multigrid
        # levels: 16^3, where launches and one wave's latency are all there is
        dict(name="matmult-f64-16", kind="matmult", mx=16, my=16, mz=16, bits=64, mesh="perturbed", eta="random"),
        # a medium box whose sides fit no tile, on a deformed mesh
        dict(name="matmult-f64-ragged", kind="matmult", mx=45, my=37, mz=29, bits=64, mesh="perturbed", eta="random"),
        # the headline MatMult: 64^3 with sinker viscosity
        dict(name="matmult-f64-64", kind="matmult", mx=64, my=64, mz=64, bits=64, mesh="box", eta="sinker"),
        # the same operator in FP32, the work of an FP32 V-cycle's smoother
        dict(name="matmult-f32-64", kind="matmult", mx=64, my=64, mz=64, bits=32, mesh="box", eta="sinker"),
        # the finest level of the large solve: 128^3, layers at contrast 1e6
        dict(name="matmult-f64-128", kind="matmult", mx=128, my=128, mz=128, bits=64, mesh="box", eta="layers"),
        # the saddle-point operator of an outer FGMRES on a rift-shaped box
        dict(name="stokes-96x96x48", kind="stokes", mx=96, my=96, mz=48, mesh="box", eta="layers"),
        # gradient and divergence apart, as a segregated or fieldsplit solver
        # calls them
        dict(name="a12-a21-64x48x40", kind="coupling", mx=64, my=48, mz=40, mesh="perturbed"),
        # one Picard step's coefficients: power-law viscosity of the current
        # velocity, installed in the operator, and the new Jacobi diagonal
        dict(name="picard-coefficients-48", kind="picard", mx=48, my=48, mz=48, mesh="perturbed", nexp=3.0),
        # marker viscosity to the quadrature points after an advection step,
        # 3 x 3 x 3 jittered points per element in element order
        dict(name="points-40x40x24", kind="points", mx=40, my=40, mz=24, mesh="box", per=3, shuffled=False),
        # one smoother call of an FP32 V-cycle: Chebyshev(3) from a nonzero guess
        dict(name="smooth-f32-48x48x32", kind="smooth", mx=48, my=48, mz=32, levels=4, bits=32, its=3),
        # the preconditioner of the velocity block: an FP64 V-cycle, 64^3 to 4^3
        dict(name="vcycle-f64-64", kind="vcycle", mx=64, my=64, mz=64, levels=5, eta="sinker", its=3),
        # many small independent boxes in one batched MatMult
        dict(name="batch-f64-32-boxes", kind="batch", boxes=32, lo=4, hi=24, bits=64, shapes=7),
    ]


def _side(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi, most):
    while True:
        m = [_side(rng, lo, hi) for _ in range(3)]
        if m[0] * m[1] * m[2] <= most:
            return dict(mx=m[0], my=m[1], mz=m[2])


def draw(rng):
    kind = rng.choice(("matmult", "matmult", "matmult", "stokes", "coupling", "picard", "points", "smooth", "vcycle",
                       "batch"))
    mesh = rng.choice(("box", "perturbed"))
    if kind == "matmult":
        return dict(kind=kind, **_box(rng, 8, 128, MAX_ELEMENTS), bits=rng.choice((64, 64, 32)), mesh=mesh,
                    eta=rng.choice(("random", "sinker", "layers")))
    if kind == "stokes":
        return dict(kind=kind, **_box(rng, 8, 96, 96 * 96 * 48), mesh=mesh, eta=rng.choice(("random", "layers")))
    if kind == "coupling":
        return dict(kind=kind, **_box(rng, 8, 96, 200000), mesh=mesh)
    if kind == "picard":
        return dict(kind=kind, **_box(rng, 8, 80, 150000), mesh=mesh, nexp=rng.choice((1.5, 2.0, 3.0, 3.5)))
    if kind == "points":
        return dict(kind=kind, **_box(rng, 8, 64, 60000), mesh=mesh, per=rng.choice((2, 3)), shuffled=rng.random() < 0.3)
    if kind == "batch":
        lo = rng.randint(3, 8)
        return dict(kind=kind, boxes=rng.randint(8, 40), lo=lo, hi=lo + rng.randint(4, 16), bits=rng.choice((64, 32)),
                    shapes=rng.randint(0, 10 ** 6))
    # hierarchies: a coarsest box of 3 to 5 elements a side, 3 to 5 levels
    while True:
        levels = rng.randint(3, 5)
        m = [rng.randint(3, 5) << (levels - 1) for _ in range(3)]
        if m[0] * m[1] * m[2] <= 64 ** 3:
            break
    c = dict(kind=kind, mx=m[0], my=m[1], mz=m[2], levels=levels, its=rng.choice((2, 3, 4)))
    return dict(c, bits=rng.choice((32, 64))) if kind == "smooth" else dict(c, eta=rng.choice(("random", "sinker")))


# ---- inputs ------------------------------------------------------------------

def _gen(seed, k):
    return torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) + k)


def _uniform(seed, k, n, lo=-1.0, hi=1.0):
    return torch.rand(n, generator=_gen(seed, k), device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _mesh(case, seed):
    """Node coordinates on the host: the unit box, or its inner nodes moved by
    up to a tenth of the node spacing."""
    m = case["mx"], case["my"], case["mz"]
    x = F.box_coords(*m)
    return F.perturb_interior(x, *m, 0.1, np.random.default_rng(seed)) if case.get("mesh") == "perturbed" else x


def _viscosity(m, kind, seed):
    """Quadrature-point viscosity on the device, element-major."""
    mx, my, mz = m
    if kind == "random":
        return 10.0 ** _uniform(seed, 11, 27 * mx * my * mz, -2.0, 2.0)
    rng = np.random.default_rng(seed)
    gx, gy, gz = (torch.from_numpy(a).cuda() for a in F.box_qp_axes(*m))
    gx, gy, gz = gx[None, None, :, None, None, :], gy[None, :, None, None, :, None], gz[:, None, None, :, None, None]
    if kind == "sinker":  # 32 spheres at 1e4 in a background of 1
        eta = torch.ones(mz, my, mx, 3, 3, 3, dtype=torch.float64, device="cuda")
        for c, r in zip(rng.uniform(0.0, 1.0, (32, 3)), rng.uniform(0.05, 0.12, 32)):
            eta[(gx - c[0]) ** 2 + (gy - c[1]) ** 2 + (gz - c[2]) ** 2 <= r * r] = 1e4
    elif kind == "layers":  # 1e3 / 1e1 / 1e-3 from the base up, weak ellipsoids at 1e-3
        z = torch.where(gz < 1 / 3, 1e3, torch.where(gz < 2 / 3, 1e1, 1e-3)).to(torch.float64)
        eta = z.expand(mz, my, mx, 3, 3, 3).contiguous()
        for c, a in zip(rng.uniform(0.0, 1.0, (24, 3)), rng.uniform(0.03, 0.1, (24, 3))):
            eta[((gx - c[0]) / a[0]) ** 2 + ((gy - c[1]) / a[1]) ** 2 + ((gz - c[2]) / a[2]) ** 2 <= 1.0] = 1e-3
    else:  # "smooth": one decade either way over the box
        k = rng.integers(1, 4, 3)
        eta = 10.0 ** (torch.sin(math.pi * k[0] * gx) * torch.sin(math.pi * k[1] * gy) * torch.cos(math.pi * k[2] * gz))
    return eta.reshape(-1).contiguous()


def _boundary(case):
    m = case["mx"], case["my"], case["mz"]
    return F.rift_bc(*m)[0] if case["kind"] == "stokes" else F.dirichlet_all_faces(*m)


def _operator(case, coords, eta, bc, cls=MatA11MF):
    op = cls(case["mx"], case["my"], case["mz"])
    op.set_coordinates(coords)
    if eta is not None:
        op.set_viscosity_device(TensorArray(eta))
    op.set_dirichlet(bc)
    op.is_setup = True
    return op


def _sizes(case):
    m = case["mx"], case["my"], case["mz"]
    return 3 * F.nnodes(*m), m[0] * m[1] * m[2]


def _hierarchy(case, seed, bits, eta):
    m = case["mx"], case["my"], case["mz"]
    mg = GMG(*m, case["levels"])
    mg.set_coordinates(F.box_coords(*m))
    mg.set_viscosity(case["levels"] - 1, _viscosity(m, eta, seed).cpu().numpy())
    mg.coarsen_viscosity("qp-arithmetic")
    mg.set_dirichlet_all_faces()
    mg.setup(default_options(smoother_precision=bits, pre_its=case["its"], post_its=case["its"]))
    return mg


def _points(case, seed):
    """A jittered lattice of points per element, their element indices and a
    viscosity each; shuffled: in no element order, as after many steps."""
    m, per = (case["mx"], case["my"], case["mz"]), case["per"]
    E, n = m[0] * m[1] * m[2], per ** 3
    g = -1.0 + (2.0 / per) * (torch.arange(per, device="cuda", dtype=torch.float64) + 0.5)
    lat = torch.stack(torch.meshgrid(g, g, g, indexing="ij"), -1).reshape(n, 3)
    xi = lat.repeat(E, 1) + _uniform(seed, 21, 3 * n * E, -0.5 / per, 0.5 / per).view(-1, 3)
    elem = torch.arange(E, device="cuda").repeat_interleave(n)
    val = 10.0 ** _uniform(seed, 22, n * E, -2.0, 2.0)
    if case["shuffled"]:
        p = torch.randperm(n * E, generator=_gen(seed, 23), device="cuda")
        xi, elem, val = xi[p], elem[p], val[p]
    return elem.contiguous(), xi.reshape(-1).contiguous(), val.contiguous()


SMOOTH_EIGS = (0.6, 3.3)  # bounds that a program carries over from an earlier set-up


def _batch_boxes(case, seed):
    """One case dict per box of a batch (uneven sides, the same for every seed)."""
    rng = np.random.default_rng(case["shapes"])
    return [dict(kind="matmult", mx=int(a), my=int(b), mz=int(c), mesh="perturbed", eta="random", bits=case["bits"])
            for a, b, c in rng.integers(case["lo"], case["hi"] + 1, (case["boxes"], 3))]


class State:
    def __init__(self, kind):
        self.kind = kind
        self.batch = None

    def __del__(self):
        if self.batch is not None:
            self.batch.destroy()


def _dtype(case):
    return torch.float32 if case["bits"] == 32 else torch.float64


def prepare(case, seed):
    s = State(case["kind"])
    if s.kind == "batch":
        boxes = _batch_boxes(case, seed)
        s.ops, s.x, s.y = [], [], []
        for k, c in enumerate(boxes):
            sd = seed * 1000 + k
            n = _sizes(c)[0]
            s.ops.append(_operator(c, _mesh(c, sd), _viscosity((c["mx"], c["my"], c["mz"]), "random", sd), _boundary(c)))
            s.x.append(TensorArray(_uniform(sd, 1, n).to(_dtype(c))))
            s.y.append(TensorArray(torch.empty_like(s.x[-1].tensor)))
        s.bits = case["bits"]
        s.batch = BatchA11(s.ops)
        torch.cuda.synchronize()
        return s
    n, E = _sizes(case)
    m = case["mx"], case["my"], case["mz"]
    if s.kind == "smooth":
        s.level, s.its = case["levels"] - 1, case["its"]
        s.mg = _hierarchy(case, seed, case["bits"], "smooth")
        s.mg.set_eigs(s.level, *SMOOTH_EIGS)
        s.b = TensorArray(_uniform(seed, 1, n).to(_dtype(case)))
        s.x0 = _uniform(seed, 2, n).to(_dtype(case))
        s.x = TensorArray(s.x0.clone())
    elif s.kind == "vcycle":
        s.mg = _hierarchy(case, seed, 64, case["eta"])
        s.b = TensorArray(_uniform(seed, 1, n))
        s.x = TensorArray(torch.empty_like(s.b.tensor))
    elif s.kind == "points":
        s.op = _operator(case, _mesh(case, seed), None, _boundary(case))
        s.elem, s.xi, s.val = (TensorArray(t) for t in _points(case, seed))
        s.eta = TensorArray(torch.empty(27 * E, dtype=torch.float64, device="cuda"))
    elif s.kind == "picard":
        # the operator holds the last step's viscosity; the new one overwrites it
        s.op = _operator(case, _mesh(case, seed), torch.ones(27 * E, dtype=torch.float64, device="cuda"), _boundary(case))
        s.u = TensorArray(_uniform(seed, 1, n))
        s.B = TensorArray(10.0 ** _uniform(seed, 2, 27 * E))
        s.nexp = case["nexp"]
        s.eta = TensorArray(torch.empty(27 * E, dtype=torch.float64, device="cuda"))
        s.d = TensorArray(torch.empty(n, dtype=torch.float64, device="cuda"))
    elif s.kind == "coupling":
        s.op = _operator(case, _mesh(case, seed), None, _boundary(case), MatStokesMF)
        s.p, s.u = TensorArray(_uniform(seed, 1, 4 * E)), TensorArray(_uniform(seed, 2, n))
        s.yu = TensorArray(torch.empty(n, dtype=torch.float64, device="cuda"))
        s.yp = TensorArray(torch.empty(4 * E, dtype=torch.float64, device="cuda"))
    else:
        cls = MatStokesMF if s.kind == "stokes" else MatA11MF
        s.op = _operator(case, _mesh(case, seed), _viscosity(m, case["eta"], seed), _boundary(case), cls)
        x = _uniform(seed, 1, n + (4 * E if s.kind == "stokes" else 0))
        s.x = TensorArray(x.to(_dtype(case)) if s.kind == "matmult" else x)
        s.y = TensorArray(torch.empty_like(s.x.tensor))
    torch.cuda.synchronize()
    return s


def run(s):
    if s.kind == "matmult":
        s.op.mult(s.x, s.y)
        return s.y.tensor
    if s.kind == "stokes":
        s.op.mult_stokes(s.x, s.y)
        return s.y.tensor
    if s.kind == "coupling":
        s.op.mult_a12(s.p, s.yu)
        s.op.mult_a21(s.u, s.yp)
        return {"yu": s.yu.tensor, "yp": s.yp.tensor}
    if s.kind == "picard":
        s.op.powerlaw_viscosity(s.u, s.B, s.nexp, 1e-3, 1e3, s.eta)
        s.op.set_viscosity_device(s.eta)
        s.op.get_diagonal(s.d)
        return {"eta": s.eta.tensor, "diagonal": s.d.tensor}
    if s.kind == "points":
        s.op.project_points(s.elem, s.xi, s.val, s.eta)
        return s.eta.tensor
    if s.kind == "smooth":
        s.x.tensor.copy_(s.x0)  # the smoother works in place: the same guess for each pass
        s.mg.smooth(s.level, s.b, s.x, s.its, True)
        return s.x.tensor
    if s.kind == "vcycle":
        s.mg.vcycle(s.b, s.x)
        return s.x.tensor
    s.batch.mult(s.x, s.y, s.bits)
    return [y.tensor for y in s.y]


# ---- what a pass cannot do without -------------------------------------------

def _matmult_work(case):
    n, E = _sizes(case)
    return (case["bits"] // 8) * (3 * n + 27 * E), A11_FLOPS * E


def work(case):
    kind = case["kind"]
    if kind == "batch":
        w = [_matmult_work(c) for c in _batch_boxes(case, 0)]
        return {"bytes": sum(a for a, _ in w), "flops": sum(b for _, b in w)}
    n, E = _sizes(case)
    if kind == "matmult":
        b, f = _matmult_work(case)
    elif kind == "stokes":  # also p in, B^T u out
        b, f = 8 * (3 * n + 27 * E + 8 * E), (A11_FLOPS + 1200) * E
    elif kind == "coupling":  # coordinates twice, u in, y out, p in, yp out
        b, f = 8 * (4 * n + 8 * E), 2 * 5000 * E
    elif kind == "picard":  # coordinates, u, B in; eta out; its operator copies out; coordinates and eta in, diagonal out
        b, f = 8 * (2 * n + 54 * E) + 12 * 27 * E + 8 * (2 * n + 27 * E), 20000 * E
    elif kind == "points":  # the points in (element, xi, value), eta out
        b, f = 40 * E * case["per"] ** 3 + 8 * 27 * E, E * (40 * case["per"] ** 3 + 800)
    elif kind == "smooth":  # its + 1 MatMults and the update streams
        w = case["bits"] // 8
        b, f = w * ((case["its"] + 1) * (3 * n + 27 * E) + 4 * n), (case["its"] + 1) * A11_FLOPS * E
    else:  # per level 2 its + 2 MatMults; the coarser levels add 1/7
        b, f = 8 * (2 * case["its"] + 2) * (3 * n + 27 * E) * 8 // 7, (2 * case["its"] + 2) * A11_FLOPS * E * 8 // 7
    return {"bytes": b, "flops": f}


# ---- the same outputs in plain 64-bit torch ------------------------------------

_S = math.sqrt(0.6)
_GP = (-_S, 0.0, _S)
_N1 = [[0.5 * x * (x - 1), (1 + x) * (1 - x), 0.5 * x * (x + 1)] for x in _GP]
_D1 = [[x - 0.5, -2 * x, x + 0.5] for x in _GP]
_W1 = (5 / 9, 8 / 9, 5 / 9)


def _tables():
    """Basis values [27 qp, 27 nodes], reference gradients [27, 3, 27], weights [27]."""
    N, D, W = (torch.tensor(t, dtype=torch.float64, device="cuda") for t in (_N1, _D1, _W1))
    ein = lambda a, b, c: torch.einsum("ai,bj,ck->cbakji", a, b, c).reshape(27, 27)  # noqa: E731
    G = torch.stack([ein(D, N, N), ein(N, D, N), ein(N, N, D)], 1)
    w = (W[:, None, None] * W[None, :, None] * W[None, None, :]).reshape(27)
    return ein(N, N, N), G, w


class _Exact:
    """Element sums over chunks of elements: geometry at the quadrature points
    by straight 27-term sums, scatter by index_add."""

    def __init__(self, case, coords, eta=None, bc=None):
        self.m = case["mx"], case["my"], case["mz"]
        self.E = self.m[0] * self.m[1] * self.m[2]
        self.x = torch.from_numpy(coords).cuda().view(-1, 3)
        self.eta = None if eta is None else eta.view(self.E, 27)
        self.bc = torch.from_numpy(np.asarray(bc, dtype=bool)).cuda()
        self.N, self.G, self.w = _tables()

    def chunks(self, step=16384):
        mx, my, _ = self.m
        X, Y = 2 * mx + 1, 2 * my + 1
        k, j, i = (t.reshape(-1) for t in torch.meshgrid(*[torch.arange(3, device="cuda")] * 3, indexing="ij"))
        for e0 in range(0, self.E, step):
            e = torch.arange(e0, min(e0 + step, self.E), device="cuda")
            ei, ej, ek = e % mx, (e // mx) % my, e // (mx * my)
            nid = (2 * ei[:, None] + i) + X * ((2 * ej[:, None] + j) + Y * (2 * ek[:, None] + k))
            xe = self.x[nid]  # [e, 27, 3]
            J = self.ref_grad(xe)  # [e, 27 qp, 3 (xi), 3 (x)]
            a, b, c = J[:, :, 0], J[:, :, 1], J[:, :, 2]
            det = (a * torch.linalg.cross(b, c)).sum(-1)
            inv = torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)], 2)
            inv = inv / det[..., None, None]  # [e, q, j, d] = d xi_j / d x_d
            yield slice(e0, e0 + len(e)), nid, xe, inv, det * self.w

    def ref_grad(self, v):
        """[e, 27, c] nodal values -> [e, 27 qp, 3, c] reference gradients."""
        e, _, c = v.shape
        return (self.G.view(81, 27) @ v.permute(1, 0, 2).reshape(27, e * c)).view(27, 3, e, c).permute(2, 0, 1, 3)

    def to_nodes(self, f):
        """transpose of ref_grad: [e, 27 qp, 3, c] -> [e, 27, c]"""
        e, c = f.shape[0], f.shape[3]
        return (self.G.view(81, 27).T @ f.permute(1, 2, 0, 3).reshape(81, e * c)).view(27, e, c).permute(1, 0, 2)

    def pressure_basis(self, xe):
        xq = (self.N @ xe.permute(1, 0, 2).reshape(27, -1)).view(27, -1, 3).permute(1, 0, 2)  # [e, q, 3]
        L = torch.stack([xe[:, 14, 0] - xe[:, 12, 0], xe[:, 16, 1] - xe[:, 10, 1], xe[:, 22, 2] - xe[:, 4, 2]], -1)
        rel = (xq - xe.mean(1, keepdim=True)) / L[:, None]
        return torch.cat([torch.ones_like(rel[..., :1]), rel], -1)  # [e, q, 4]

    def stokes(self, u=None, p=None):
        """(A11 mask(u) + A12 p on free rows and the boundary rows apart, A21 mask(u))"""
        um = None if u is None else torch.where(self.bc, 0.0, u).view(-1, 3)
        yu = torch.zeros_like(self.x)
        yp = torch.zeros(self.E, 4, dtype=torch.float64, device="cuda")
        for sl, nid, xe, inv, wdet in self.chunks():
            s = torch.zeros(len(nid), 27, 3, 3, dtype=torch.float64, device="cuda")
            if um is not None:
                g = inv.transpose(2, 3) @ self.ref_grad(um[nid])  # [e, q, d, c] = d u_c / d x_d
                if self.eta is not None:
                    s += (self.eta[sl] * wdet)[..., None, None] * (g + g.transpose(2, 3))
                div = g.diagonal(dim1=2, dim2=3).sum(-1)
            P = self.pressure_basis(xe) if p is not None or self.eta is None else None
            if p is not None:
                s -= (wdet * (P * p.view(-1, 4)[sl][:, None]).sum(-1))[..., None, None] * torch.eye(3, device="cuda", dtype=torch.float64)
            if P is not None and um is not None:
                yp[sl] = -(P * (wdet * div)[..., None]).sum(1)
            yu.index_add_(0, nid.reshape(-1), self.to_nodes(inv @ s).reshape(-1, 3))
        return yu.reshape(-1), yp.reshape(-1)

    def a11(self, u):
        return torch.where(self.bc, u, self.stokes(u)[0])

    def diagonal(self, eta):
        d = torch.zeros_like(self.x)
        for sl, nid, xe, inv, wdet in self.chunks(8192):
            g = torch.einsum("eqjd,qjn->eqnd", inv, self.G)
            s = (eta.view(self.E, 27)[sl] * wdet)[..., None, None]
            d.index_add_(0, nid.reshape(-1), (s * (g.square().sum(-1, keepdim=True) + g.square())).sum(1).reshape(-1, 3))
        return torch.where(self.bc, 1.0, d.reshape(-1))

    def powerlaw(self, u, B, nexp, lo, hi):
        eta = torch.empty(self.E, 27, dtype=torch.float64, device="cuda")
        for sl, nid, xe, inv, wdet in self.chunks():
            g = inv.transpose(2, 3) @ self.ref_grad(u.view(-1, 3)[nid])
            e2 = (0.5 * (g + g.transpose(2, 3))).square().sum((2, 3))
            eta[sl] = B.view(-1, 27)[sl] * torch.sqrt(0.5 * e2).clamp_min(1e-17) ** (1.0 / nexp - 1.0)
        return eta.clamp(lo, hi).reshape(-1)


def _exact_points(case, seed):
    elem, xi, val = _points(case, seed)
    mx, my, mz = case["mx"], case["my"], case["mz"]
    X, Y, Z = 2 * mx + 1, 2 * my + 1, 2 * mz + 1
    xi = xi.view(-1, 3)
    f = [torch.stack([0.5 * (1 - xi[:, d]), torch.ones_like(val), 0.5 * (1 + xi[:, d])], 1) for d in range(3)]
    e = torch.arange(mx * my * mz, device="cuda")
    base = 2 * (e % mx) + X * (2 * ((e // mx) % my) + Y * 2 * (e // (mx * my)))
    A, B = (torch.zeros(X * Y * Z, dtype=torch.float64, device="cuda") for _ in range(2))
    for n in range(27):
        i, j, k = n % 3, n // 3 % 3, n // 9
        w = torch.ones_like(val) if (i | j | k) & 1 else f[0][:, i] * f[1][:, j] * f[2][:, k]
        node = base[elem] + i + X * (j + Y * k)
        A.index_add_(0, node, w * val)
        B.index_add_(0, node, w)
    nodal = A / B
    ne = torch.stack([nodal[base + n % 3 + X * (n // 3 % 3 + Y * (n // 9))] for n in range(27)], 1)
    g = torch.tensor(_GP, dtype=torch.float64, device="cuda")
    q1 = torch.stack([0.5 * (1 - g), 0.5 * (1 + g)], 1)  # [gp, side]
    Q = torch.einsum("ai,bj,ck->cbakji", q1, q1, q1).reshape(27, 8)
    v = ne[:, [0, 2, 6, 8, 18, 20, 24, 26]] @ Q.T
    return torch.minimum(torch.maximum(v, ne.min(1, keepdim=True).values), ne.max(1, keepdim=True).values).reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "vcycle":
        return None
    if kind == "points":
        return _exact_points(case, seed)
    if kind == "batch":
        out = []
        for k, c in enumerate(_batch_boxes(case, seed)):
            sd = seed * 1000 + k
            ex = _Exact(c, _mesh(c, sd), _viscosity((c["mx"], c["my"], c["mz"]), "random", sd), _boundary(c))
            out.append(ex.a11(_uniform(sd, 1, _sizes(c)[0]).to(_dtype(c)).double()))
        return out
    n, E = _sizes(case)
    m = case["mx"], case["my"], case["mz"]
    if kind == "smooth":
        eta = _viscosity(m, "smooth", seed)
        ex = _Exact(case, F.box_coords(*m), eta, _boundary(case))
        d = ex.diagonal(eta)
        b, x = (_uniform(seed, k, n).to(_dtype(case)).double() for k in (1, 2))
        emin, emax = SMOOTH_EIGS
        scale = 2.0 / (emax + emin)
        mu = 1.0 / (1.0 - scale * emin)
        c = [1.0, mu]
        p = [x, x + scale * (b - ex.a11(x)) / d]
        for _ in range(case["its"]):
            c.append(2.0 * mu * c[-1] - c[-2])
            om = 2.0 * mu * c[-2] / c[-1]
            p.append(om * scale * (b - ex.a11(p[-1])) / d + (1.0 - om) * p[-2] + om * p[-1])
        return p[-1]
    if kind == "coupling":
        ex = _Exact(case, _mesh(case, seed), None, _boundary(case))
        yu = ex.stokes(p=_uniform(seed, 1, 4 * E))[0]
        return {"yu": torch.where(ex.bc, 0.0, yu), "yp": ex.stokes(u=_uniform(seed, 2, n))[1]}
    if kind == "picard":
        ex = _Exact(case, _mesh(case, seed), None, _boundary(case))
        eta = ex.powerlaw(_uniform(seed, 1, n), 10.0 ** _uniform(seed, 2, 27 * E), case["nexp"], 1e-3, 1e3)
        return {"eta": eta, "diagonal": ex.diagonal(eta)}
    ex = _Exact(case, _mesh(case, seed), _viscosity(m, case["eta"], seed), _boundary(case))
    x = _uniform(seed, 1, n + (4 * E if kind == "stokes" else 0))
    if kind == "matmult":
        return ex.a11(x.to(_dtype(case)).double())
    yu, _ = ex.stokes(x[:n], x[n:])
    return torch.cat([torch.where(ex.bc, x[:n], yu), ex.stokes(x[:n], x[n:])[1]])
