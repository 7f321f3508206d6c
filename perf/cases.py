"""The work a user of yeti_amd has it do, as cases that can be timed and checked.

Every case is a cantilever of the repository's workloads: a 10 x 1 x 1 NURBS box, face x = 0
clamped, a traction in z on the face x = 10, interior control points jittered by 5 % of an
element, weights in [0.8, 1.2]. Sizes are elements per direction, ``p0 p1 p2`` the degrees and
``ng`` the Gauss points per direction. The kinds:

  assemble    COO triplets and F of a resident model (``Assembler.run_coo``)
  reassemble  design update: new control points, then the values and F again
  csr         CSR values of K + K^T from the COO values, and one product with a vector
  apply       the matrix-free product K x in FP64 or FP32, inside every iterative solve
  mass        the consistent mass matrix (COO triplets) of a modal analysis
  vib         d(eigenvalue)/d(control points) of a set of modes
  shape       work gradients of a state and its adjoints, volume and its gradient
  compliance  one step of a shape optimisation: J and dJ/dX through autograd, solve included
  serve       a group of solve requests of mixed sizes through the batched server

``exact`` restates what each of them computes in plain 64-bit torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from yeti_amd.assembly import Assembler
from yeti_amd.gradient import CompliancePatch, compliance
from yeti_amd.matfree import F32, F64, MatrixFree
from yeti_amd.serving import Request, SolveServer, request_stream
from yeti_amd.solver import StiffnessCSR

LENGTH = (10.0, 1.0, 1.0)
E, NU, RHO, TRACTION = 210000.0, 0.3, 7.8e-9, -1.0


def _case(kind, nel, p, ng=None, **more):
    p = (p, p, p) if isinstance(p, int) else p
    return dict(kind=kind, n0=nel[0], n1=nel[1], n2=nel[2], p0=p[0], p1=p[1], p2=p[2],
                ng=ng if ng is not None else max(p) + 1, **more)


def listed():
    return [
        # the smallest model of the repository's tests and benchmark: a call that is all latency
        dict(name="assemble_16x4x4_p2", **_case("assemble", (16, 4, 4), 2)),
        # the benchmark's assembly: 262,144 elements, 4.9e9 COO entries
        dict(name="assemble_64x64x64_p3", **_case("assemble", (64, 64, 64), 3)),
        # a refined model whose directions have different degrees, as refining a coarse beam gives
        dict(name="assemble_45x14x11_p231", **_case("assemble", (45, 14, 11), (2, 3, 1))),
        # the inner step of a design loop at the highest degree: indices are known, values change
        dict(name="reassemble_23x18x13_p4", **_case("reassemble", (23, 18, 13), 4)),
        # the assembled operator of an iterative solve, refreshed and used
        dict(name="csr_45x40x33_p3", **_case("csr", (45, 40, 33), 3)),
        # the operator of the large mixed-precision solve: 6.6M unknowns
        dict(name="apply_f32_128x128x128_p2", **_case("apply", (128, 128, 128), 2, bits=32)),
        # an ordinary odd-sized FP64 product
        dict(name="apply_f64_37x29x41_p3", **_case("apply", (37, 29, 41), 3, bits=64)),
        # modal analysis of an ordinary model
        dict(name="mass_61x53x47_p2", **_case("mass", (61, 53, 47), 2)),
        # frequency gradient of four modes, an ordinary odd-sized model
        dict(name="vib_33x29x26_p3", **_case("vib", (33, 29, 26), 3, modes=4)),
        # gradients of an optimisation iteration: two adjoint fields and the volume
        dict(name="shape_47x31x22_p2", **_case("shape", (47, 31, 22), 2, adjoints=2)),
        # one step of the 32^3 shape optimisation, assembly, solve and gradient
        dict(name="compliance_32x32x32_p2", **_case("compliance", (32, 32, 32), 2)),
        # requests of 4 to 48 elements per direction and degrees 2 to 4, all at once
        dict(name="serve_24_mixed", kind="serve", requests=24, lo=4, hi=48, stream=20261202, precision="mixed"),
    ]


# the largest number of elements that draw() gives, by kind and degree 1 .. 4: the listed sizes
# and their like
_MOST = {
    "assemble": (262144, 262144, 65536, 8192),
    "general": (32768, 16384, 8192, 8192),
    "reassemble": (262144, 131072, 32768, 5400),
    "csr": (262144, 131072, 59400, 8192),
    "apply": (2097152, 2097152, 262144, 65536),
    "mass": (262144, 152000, 65536, 8192),
    "vib": (65536, 49152, 24882, 8192),
    "shape": (65536, 32768, 16384, 5400),
    "compliance": (32768, 32768, 4096, 512),
}


def draw(rng):
    kind = rng.choice(list(_MOST) + ["serve"])
    if kind == "serve":
        hi = rng.randint(8, 40)
        return dict(kind="serve", requests=rng.randint(1, 20), lo=4, hi=hi, stream=rng.randrange(1 << 30),
                    precision=rng.choice(["mixed", "mixed", "fp64"]))
    more = {}
    if kind == "general":
        # unequal degrees, or more Gauss points than p + 1
        p = tuple(rng.randint(1, 3) for _ in range(3))
        ng = max(p) + (2 if p[0] == p[1] == p[2] else 1)
    elif kind == "compliance":
        p, ng = rng.choice([1, 2, 2, 3]), None
    else:
        p, ng = rng.choice([1, 2, 2, 3, 3, 4]), None
    top = max(p) if isinstance(p, tuple) else p
    ne = math.exp(rng.uniform(math.log(16), math.log(_MOST[kind][top - 1])))
    # aspect ratios from a cube to a beam
    s = [math.exp(rng.uniform(0.0, 1.1)), math.exp(rng.uniform(-0.5, 0.5)), 1.0]
    f = (ne / (s[0] * s[1] * s[2])) ** (1.0 / 3.0)
    nel = [max(1, int(f * x)) for x in s]
    if kind == "apply":
        more["bits"] = rng.choice([32, 64])
    elif kind == "vib":
        more["modes"] = rng.choice([1, 2, 4, 5])
    elif kind == "shape":
        more["adjoints"] = rng.choice([1, 2, 3])
    return _case("assemble" if kind == "general" else kind, nel, p, ng, **more)


# ---- models ------------------------------------------------------------------------------
def _dims(case):
    nel = (case["n0"], case["n1"], case["n2"])
    p = (case["p0"], case["p1"], case["p2"])
    return nel, p, case["ng"]


def _knots(n, p):
    return np.concatenate([np.zeros(p + 1), np.arange(1, n) / n, np.ones(p + 1)])


def _net(nel, p, seed):
    """Control points (3, ncp), weights (ncp) and grid sizes; xi fastest."""
    nc = [nel[d] + p[d] for d in range(3)]
    g = []
    for d in range(3):
        U = _knots(nel[d], p[d])
        g.append(np.array([U[i + 1:i + p[d] + 1].mean() for i in range(nc[d])]) * LENGTH[d])
    rng = np.random.default_rng(seed)
    X = np.empty((nc[2], nc[1], nc[0], 3))
    X[..., 0], X[..., 1], X[..., 2] = g[0], g[1][:, None], g[2][:, None, None]
    h = np.array([LENGTH[d] / nel[d] for d in range(3)])
    X[1:-1, 1:-1, 1:-1] += (rng.random((max(nc[2] - 2, 0), max(nc[1] - 2, 0), max(nc[0] - 2, 0), 3)) - 0.5) * 0.1 * h
    w = 0.8 + 0.4 * rng.random(nc[0] * nc[1] * nc[2])
    return np.asfortranarray(X.reshape(-1, 3).T), w, nc


def _connectivity(nel, p, nc):
    """0-based control points per element (ne, nnode); local node 0 is the highest corner."""
    idx = []
    for d in range(3):
        idx.append(np.arange(nel[d], dtype=np.int32)[:, None] + p[d] - np.arange(p[d] + 1, dtype=np.int32)[None, :])
    i0 = idx[0][None, None, :, None, None, :]
    i1 = idx[1][None, :, None, None, :, None] * np.int32(nc[0])
    i2 = idx[2][:, None, None, :, None, None] * np.int32(nc[0] * nc[1])
    return (i0 + i1 + i2).reshape(nel[0] * nel[1] * nel[2], -1)


def _model(case, seed):
    """The arguments of sys_linmat_lindef_static for the case's cantilever, by name."""
    nel, p, ng = _dims(case)
    X, w, nc = _net(nel, p, seed)
    ien = _connectivity(nel, p, nc)
    ne, ncp = ien.shape[0], X.shape[1]
    e0 = np.tile(np.arange(nel[0], dtype=np.int32), nel[1] * nel[2])
    e1 = np.tile(np.repeat(np.arange(nel[1], dtype=np.int32), nel[0]), nel[2])
    e2 = np.repeat(np.arange(nel[2], dtype=np.int32), nel[0] * nel[1])
    face0 = (np.arange(nc[1] * nc[2], dtype=np.int32) * nc[0] + 1).astype(np.int32)
    fixed = np.zeros((ncp, 3), bool)
    fixed[face0 - 1] = True
    free = np.where(~fixed.reshape(-1))[0] + 1
    ind = np.zeros(3 * ncp, np.int32)
    ind[:free.size] = free
    loaded = (np.where(e0 == nel[0] - 1)[0] + 1).astype(np.int32)
    nd = 3 * ien.shape[1]
    U = [_knots(nel[d], p[d]) for d in range(3)]
    return dict(
        activeElement=np.ones(ne, np.int32), nb_data=float(ne * nd * (nd + 1) / 2), COORDS3D=X,
        IEN=(ien + 1).ravel(), nb_elem_patch=np.array([ne], np.int32),
        Nkv=np.asfortranarray(np.array([[u.size] for u in U], np.int32)), Ukv=np.concatenate(U),
        Nijk=np.asfortranarray(np.stack([e0 + p[0] + 1, e1 + p[1] + 1, e2 + p[2] + 1])),
        weight=w[ien].ravel(), Jpqr=np.asfortranarray(np.array(p, np.int32)[:, None]), ELT_TYPE="U1",
        PROPS=np.zeros(1), JPROPS=np.array([1], np.int32),
        MATERIAL_PROPERTIES=np.asfortranarray(np.array([[E], [NU]])), n_mat_props=np.array([2], np.int32),
        RHO=np.array([RHO]), TENSOR="/THREED", indDLoad=loaded, JDLType=np.array([23], np.int32),
        ADLMAG=np.array([TRACTION]), load_target_nbelem=np.array([loaded.size], np.int32),
        load_additionalInfos=np.array([], np.float64), nb_load_additionalInfos=np.zeros(1, np.int32),
        bc_values=np.asfortranarray(np.array([[1.0, 2.0, 3.0], [0.0, 0.0, 0.0]])),
        bc_target=np.concatenate([face0, face0, face0]), bc_target_nbelem=np.full(3, face0.size, np.int32),
        ind_dof_free=ind, nb_dof_free=int(free.size), MCRD=3, NBINT=np.array([ng ** 3], np.int32),
        NNODE=np.array([ien.shape[1]], np.int32), nodal_dist=np.zeros((1, ncp), order="F"), nb_bc=3, nb_load=1,
        nb_patch=1, nb_elem=ne, nb_cp=ncp, nb_dof_tot=3 * ncp)


def _fields(case, seed, count):
    """Displacement-like fields (count, ncp, 3): bending shapes of the beam with small noise."""
    nel, p, _ = _dims(case)
    X, _, _ = _net(nel, p, seed)
    x = torch.from_numpy(np.ascontiguousarray(X.T)).cuda()
    g = torch.Generator(device="cuda").manual_seed(seed + 17)
    out = []
    for k in range(count):
        s = (k // 2 + 0.5) * math.pi / LENGTH[0]
        bend, slope = 1.0 - torch.cos(s * x[:, 0]), s * torch.sin(s * x[:, 0])
        t = 2 if k % 2 == 0 else 1
        u = torch.zeros_like(x)
        u[:, t] = bend
        u[:, 0] = -(x[:, t] - 0.5) * slope
        out.append(u + 1e-4 * torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float64) * x[:, :1] / LENGTH[0])
    return torch.stack(out)


def _requests(case, seed):
    """The requests of a serve case: sizes from the case, materials and geometry from the seed."""
    rng = np.random.default_rng(seed)
    out = []
    for r in request_stream(n=case["requests"], seed=case["stream"], nel_range=(case["lo"], case["hi"])):
        out.append(Request(r.rid, r.arrival, r.nel, r.p, float(rng.uniform(1e3, 1e5)), float(rng.uniform(0.2, 0.4)),
                           -float(rng.uniform(0.1, 10.0)), int(rng.integers(1 << 31))))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        reqs = _requests(case, seed)
        for r in reqs:
            r.model()
        return dict(case=case, requests=reqs,
                    server=SolveServer(budget_bytes=24 << 30, precision=case["precision"], batched=True))
    d = _model(case, seed)
    s = dict(case=case)
    if kind == "apply":
        s["mf"] = MatrixFree(d, precisions=F64 if case["bits"] == 64 else F64 | F32)
        g = torch.Generator(device="cuda").manual_seed(seed)
        s["x"] = torch.randn(3 * d["nb_cp"], generator=g, device="cuda", dtype=torch.float64)
        if case["bits"] == 32:
            s["x"] = s["x"].float()
        s["y"] = torch.empty_like(s["x"])
        return s
    if kind == "compliance":
        s["patch"] = CompliancePatch(d, solver="csr", rtol=1e-12)
        s["coords"] = s["patch"].coords0.to("cuda")
        return s
    s["asm"] = asm = Assembler(d)
    if kind in ("assemble", "mass"):
        s["K"], s["r"], s["c"] = asm.alloc_coo(True)
        s["F"] = torch.empty(asm.nb_dof_tot, dtype=torch.float64, device="cuda")
    elif kind == "reassemble":
        # the design that the step moves to
        X, _, _ = _net(*_dims(case)[:2], seed + 1)
        s["coords"] = torch.from_numpy(np.ascontiguousarray(X.T)).cuda()
        s["K"], _, _ = asm.alloc_coo(False)
        s["F"] = torch.empty(asm.nb_dof_tot, dtype=torch.float64, device="cuda")
    elif kind == "csr":
        s["K"], _, _ = asm.alloc_coo(False)
        asm.run_values(s["K"])
        s["csr"] = StiffnessCSR(asm)
        s["vals"] = torch.empty(s["csr"].nnz, dtype=torch.float64, device="cuda")
        s["x"] = _fields(case, seed, 1)[0].reshape(-1)
        s["y"] = torch.empty_like(s["x"])
    elif kind == "vib":
        s["modes"] = _fields(case, seed, case["modes"]).transpose(1, 2)
        s["vals"] = np.linspace(1e6, 4e7, case["modes"])
    elif kind == "shape":
        f = _fields(case, seed, 1 + case["adjoints"])
        s["sol"], s["adj"] = f[0].reshape(-1), f[1:].reshape(case["adjoints"], -1)
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "assemble":
        return s["asm"].run_coo(s["K"], s["r"], s["c"], s["F"])
    if kind == "reassemble":
        s["asm"].update_coords(s["coords"])
        return s["asm"].run_values(s["K"]), s["asm"].run_rhs(s["F"])
    if kind == "csr":
        vals = s["csr"].values(s["K"], s["vals"])
        return vals, s["csr"].spmv(vals, s["x"], s["y"])
    if kind == "apply":
        return s["mf"].apply(s["x"], s["y"])
    if kind == "mass":
        return s["asm"].run_mass(s["K"], s["r"], s["c"])
    if kind == "vib":
        return s["asm"].run_vib_grad(s["modes"], s["vals"])
    if kind == "shape":
        gint, gext = s["asm"].grad_lin_elast_work(s["sol"], s["adj"])
        vol, gvol = s["asm"].volume_grad()
        return gint, gext, vol, gvol
    if kind == "compliance":
        X = s["coords"].clone().requires_grad_(True)
        J = compliance(X, s["patch"])
        J.backward()
        return J.detach(), X.grad
    rep = s["server"].run(s["requests"], keep_solutions=True, realtime=False)
    return [rep["x"][r.rid] for r in s["requests"]]


# ---- what a pass cannot do without -------------------------------------------------------
def _counts(case):
    nel, p, ng = _dims(case)
    ne = nel[0] * nel[1] * nel[2]
    n = (p[0] + 1) * (p[1] + 1) * (p[2] + 1)
    ncp = (nel[0] + p[0]) * (nel[1] + p[1]) * (nel[2] + p[2])
    return ne, n, ncp, ng ** 3


def _nnz(case):
    nel, p, _ = _dims(case)
    t = 9
    for d in range(3):
        m = nel[d] + p[d]
        t *= sum(min(m - 1, i + p[d]) - max(0, i - p[d]) + 1 for i in range(m))
    return t


def _apply_flops(p, ng, comps):
    """Sum-factorised values and gradients of ``comps`` fields at the points, and back."""
    a, b, c = (x + 1 for x in p)
    fma = 2 * ng * a * b * c + 3 * ng * ng * b * c + 4 * ng ** 3 * c
    return 2 * 2 * fma * comps


def work(case):
    kind = case["kind"]
    if kind == "serve":
        by = fl = 0.0
        for r in _requests(case, 0):
            ncp, nq = r.nb_cp, r.nel[0] * r.nel[1] * r.nel[2] * (r.p + 1) ** 3
            # at least the set-up, about 100 iterations of the operator and the preconditioner
            by += 100 * (4 * 13 * nq + 8 * 4 * 3 * ncp)
            fl += 100 * r.nel[0] * r.nel[1] * r.nel[2] * _apply_flops((r.p,) * 3, r.p + 1, 3)
        return {"bytes": by, "flops": fl}
    ne, n, ncp, nq = _counts(case)
    p, ng = _dims(case)[1:]
    entries = ne * (9 * n * (n - 1) // 2 + 6 * n)
    model = 8.0 * 4 * ncp + 4.0 * n * ne
    grad = ne * (_apply_flops(p, ng, 1) * 6.0 + 100.0 * nq)
    if kind in ("assemble", "reassemble"):
        by = model + entries * (16.0 if kind == "assemble" else 8.0) + 24.0 * ncp
        return {"bytes": by, "flops": 9.0 * n * (n + 1) * nq * ne}
    if kind == "mass":
        return {"bytes": model + 16.0 * entries, "flops": 1.0 * n * (n + 1) * nq * ne}
    if kind == "csr":
        nnz = _nnz(case)
        return {"bytes": 8.0 * entries + 16.0 * nnz + 4.0 * nnz / 9 + 48.0 * ncp, "flops": 1.0 * entries + 2.0 * nnz}
    if kind == "apply":
        s = case["bits"] // 8
        return {"bytes": s * (13.0 * nq * ne + 6.0 * ncp), "flops": ne * (_apply_flops(p, ng, 3) + 120.0 * nq)}
    if kind == "vib":
        return {"bytes": model + 48.0 * ncp * case["modes"], "flops": grad * case["modes"]}
    if kind == "shape":
        k = case["adjoints"]
        return {"bytes": 2 * model + 24.0 * ncp * (2 * k + 2), "flops": grad * (k + 1)}
    # compliance: assembly, CSR values and some 1000 products at the least
    nnz = _nnz(case)
    return {"bytes": model + 16.0 * entries + 8.0 * nnz + 1000 * (8.0 + 4.0 / 9) * nnz,
            "flops": 9.0 * n * (n + 1) * nq * ne + 2000.0 * nnz + 2 * grad}


# ---- the same results in plain 64-bit torch ----------------------------------------------
def _basis(n, p, ng):
    """Values and first derivatives (n, ng, p + 1) of the B-splines of each element at its Gauss
    points, by the Cox-de Boor recurrence on the open uniform knots, and the weights (n, ng)."""
    U = _knots(n, p)
    x, w = np.polynomial.legendre.leggauss(ng)
    span = np.arange(n) + p
    lo, hi = U[span], U[span + 1]
    t = 0.5 * (lo + hi)[:, None] + 0.5 * (hi - lo)[:, None] * x
    N = [np.ones((n, ng))]
    low = N
    for k in range(1, p + 1):
        low = N
        N = [np.zeros((n, ng)) for _ in range(k + 1)]
        for j in range(k):
            a, b = U[span + j + 1][:, None], U[span + j + 1 - k][:, None]
            f = low[j] / (a - b)
            N[j] = N[j] + (a - t) * f
            N[j + 1] = N[j + 1] + (t - b) * f
    D = [np.zeros((n, ng)) for _ in range(p + 1)]
    for j in range(p):
        f = p * low[j] / (U[span + j + 1] - U[span + j + 1 - p])[:, None]
        D[j] = D[j] - f
        D[j + 1] = D[j + 1] + f
    # local node 0 is the highest control point
    B = np.stack(N[::-1], 2), np.stack(D[::-1], 2)
    return torch.from_numpy(B[0].copy()).cuda(), torch.from_numpy(B[1].copy()).cuda(), \
        torch.from_numpy(0.5 * (hi - lo)[:, None] * w).cuda()


class _Exact:
    """Quadrature of a model's elements in chunks: R (e, q, n), dR/dx (e, q, n, 3), dv (e, q)."""

    def __init__(self, case, X, w, E=E, nu=NU):
        self.nel, self.p, self.ng = _dims(case)
        self.tab = [_basis(self.nel[d], self.p[d], self.ng) for d in range(3)]
        self.nc = [self.nel[d] + self.p[d] for d in range(3)]
        self.ien = torch.from_numpy(_connectivity(self.nel, self.p, self.nc)).long().cuda()
        self.X = torch.from_numpy(np.ascontiguousarray(X.T)).cuda()
        self.w = torch.from_numpy(w).cuda()
        self.ne, self.n = self.ien.shape
        self.ncp = self.X.shape[0]
        self.lam, self.mu = E * nu / (1 + nu) / (1 - 2 * nu), E / 2 / (1 + nu)

    def chunks(self, extra=0):
        per = 8 * (16 * self.ng ** 3 * self.n + extra)
        step = max(1, int(2e9 // per))
        for a in range(0, self.ne, step):
            yield torch.arange(a, min(self.ne, a + step), device="cuda")

    def points(self, el):
        e = (el % self.nel[0], el // self.nel[0] % self.nel[1], el // (self.nel[0] * self.nel[1]))
        (B0, D0, w0), (B1, D1, w1), (B2, D2, w2) = [[t[e[d]] for t in self.tab[d]] for d in range(3)]

        def tensor(a, b, c):
            t = c[:, :, None, None, :, None, None] * b[:, None, :, None, None, :, None] * a[:, None, None, :, None, None, :]
            return t.reshape(el.numel(), self.ng ** 3, self.n)
        we, xe = self.w[self.ien[el]], self.X[self.ien[el]]
        N = tensor(B0, B1, B2) * we[:, None, :]
        dN = [tensor(D0, B1, B2) * we[:, None, :], tensor(B0, D1, B2) * we[:, None, :], tensor(B0, B1, D2) * we[:, None, :]]
        W = N.sum(2, keepdim=True)
        R = N / W
        G = torch.stack([(d - R * d.sum(2, keepdim=True)) / W for d in dN], 3)       # (e, q, n, m)
        J = torch.matmul(G.transpose(2, 3).contiguous(), xe[:, None].contiguous())   # dx_c / dxi_m: (e, q, m, c)
        a, b, c = J[..., 0, :], J[..., 1, :], J[..., 2, :]
        inv = torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)], -1)
        det = (a * inv[..., 0]).sum(-1)
        inv = inv / det[..., None, None]                                              # dxi_m / dx_c: (e, q, c, m)
        dR = torch.matmul(G, inv.transpose(-1, -2).contiguous())
        wq = (w2[:, :, None, None] * w1[:, None, :, None] * w0[:, None, None, :]).reshape(el.numel(), -1)
        return R, dR, wq * det

    def stiffness(self, el):
        """(e, a, k, b, l)."""
        _, dR, dv = self.points(el)
        A = (dR * dv.sqrt()[..., None, None]).reshape(el.numel(), -1, 3 * self.n)
        S = torch.bmm(A.transpose(1, 2).contiguous(), A).reshape(-1, self.n, 3, self.n, 3)
        K = self.lam * S + self.mu * S.transpose(2, 4)
        tr = S[:, :, 0, :, 0] + S[:, :, 1, :, 1] + S[:, :, 2, :, 2]
        for k in range(3):
            K[:, :, k, :, k] += self.mu * tr
        return K

    def mass(self, el):
        R, _, dv = self.points(el)
        A = R * (RHO * dv).sqrt()[..., None]
        M = torch.bmm(A.transpose(1, 2).contiguous(), A)
        K = torch.zeros(el.numel(), self.n, 3, self.n, 3, dtype=torch.float64, device="cuda")
        for k in range(3):
            K[:, :, k, :, k] = M
        return K

    def packed(self, block):
        """Upper blocks in node-pair order, diagonal halved: one row of entries per element."""
        n, at, half = self.n, [], []
        for b in range(n):
            for a in range(b + 1):
                for l in range(3):
                    for k in range(3 if a < b else l + 1):
                        at.append(((a * 3 + k) * n + b) * 3 + l)
                        half.append(0.5 if a == b and k == l else 1.0)
        at, half = torch.tensor(at, device="cuda"), torch.tensor(half, dtype=torch.float64, device="cuda")
        out = torch.empty(self.ne, at.numel(), dtype=torch.float64, device="cuda")
        for el in self.chunks(4 * (3 * n) ** 2):
            out[el[0]:el[-1] + 1] = block(el).reshape(el.numel(), -1).index_select(1, at) * half
        return out.reshape(-1)

    def load(self, traction):
        """Traction in z on the face x = 10: a quadrature over that face."""
        B0 = torch.zeros(self.p[0] + 1, dtype=torch.float64, device="cuda")
        B0[0] = 1.0
        (B1, D1, w1), (B2, D2, w2) = self.tab[1], self.tab[2]
        n1, n2, g = self.nel[1], self.nel[2], self.ng
        el = torch.arange(n1 * n2, device="cuda") * self.nel[0] + self.nel[0] - 1
        ien = self.ien[el].reshape(n2, n1, self.p[2] + 1, self.p[1] + 1, self.p[0] + 1)[..., 0]
        ien = ien.reshape(n2 * n1, -1)

        def tensor(a, b):
            t = b[:, None, :, None, :, None] * a[None, :, None, :, None, :]
            return t.reshape(n2 * n1, g * g, -1)
        we, xe = self.w[ien], self.X[ien]
        N = tensor(B1, B2) * we[:, None]
        W = N.sum(2, keepdim=True)
        R = N / W
        t = []
        for d in (tensor(D1, B2), tensor(B1, D2)):
            d = d * we[:, None]
            t.append(torch.bmm((d - R * d.sum(2, keepdim=True)) / W, xe))
        dS = torch.linalg.cross(t[0], t[1]).norm(dim=2)
        wq = (w2[:, None, :, None] * w1[None, :, None, :]).reshape(n2 * n1, -1)
        F = torch.zeros(self.ncp, 3, dtype=torch.float64, device="cuda")
        F[:, 2].index_add_(0, ien.reshape(-1), ((R * (wq * dS)[..., None]).sum(1) * traction).reshape(-1))
        return F.reshape(-1)

    def gather(self, u, el):
        return u.reshape(-1, 3)[self.ien[el]]

    def scatter(self, out, el, v):
        out.index_add_(0, self.ien[el].reshape(-1), v.reshape(-1, 3))

    def stress(self, H):
        eps = 0.5 * (H + H.transpose(-1, -2))
        s = 2 * self.mu * eps
        tr = self.lam * (H[..., 0, 0] + H[..., 1, 1] + H[..., 2, 2])
        return s + tr[..., None, None] * torch.eye(3, dtype=torch.float64, device="cuda")

    def grad(self, u, dR, el):
        """du_i/dx_k (e, q, i, k)."""
        ue = self.gather(u, el)
        return torch.matmul(ue.transpose(1, 2)[:, None].contiguous(), dR)

    def product(self, x):
        y = torch.zeros(self.ncp, 3, dtype=torch.float64, device="cuda")
        for el in self.chunks():
            _, dR, dv = self.points(el)
            s = self.stress(self.grad(x, dR, el)) * dv[..., None, None]
            self.scatter(y, el, torch.matmul(dR, s.transpose(-1, -2).contiguous()).sum(1))
        return y.reshape(-1)

    def forms(self, pairs):
        """For each (u, v, lam) of pairs: d/dX of int sigma(u) : grad v - lam rho u . v, and the
        integral of rho u . v."""
        g = [torch.zeros(self.ncp, 3, dtype=torch.float64, device="cuda") for _ in pairs]
        m = [0.0 for _ in pairs]
        for el in self.chunks():
            R, dR, dv = self.points(el)
            for k, (u, v, lam) in enumerate(pairs):
                Hu, Hv = self.grad(u, dR, el), self.grad(v, dR, el)
                su, sv = self.stress(Hu), self.stress(Hv)
                uq, vq = torch.bmm(R, self.gather(u, el)), torch.bmm(R, self.gather(v, el))
                uv = RHO * (uq * vq).sum(-1)
                m[k] = m[k] + (uv * dv).sum()
                f = ((su * Hv).sum((-1, -2)) - lam * uv)[..., None, None] * torch.eye(3, dtype=torch.float64, device="cuda")
                # T[k, m]: contracted with dR_a/dx_k gives the derivative with respect to X_am
                T = f - torch.matmul(su.transpose(-1, -2).contiguous(), Hv) - torch.matmul(sv.transpose(-1, -2).contiguous(), Hu)
                self.scatter(g[k], el, torch.matmul(dR, T * dv[..., None, None]).sum(1))
        return g, m

    def volume(self):
        vol, g = 0.0, torch.zeros(self.ncp, 3, dtype=torch.float64, device="cuda")
        for el in self.chunks():
            _, dR, dv = self.points(el)
            vol = vol + dv.sum()
            self.scatter(g, el, (dR * dv[..., None, None]).sum(1))
        return vol, g.reshape(-1)

    def assembled(self):
        """K by control point: blocks (ncp, 3, nd, 3) over the nd neighbours of the tensor grid
        (ascending control points), the neighbours (ncp, nd) and which of them exist."""
        p, nc = self.p, self.nc
        i = torch.arange(self.ncp, device="cuda")
        c = (i % nc[0], i // nc[0] % nc[1], i // (nc[0] * nc[1]))
        off = torch.cartesian_prod(*[torch.arange(-p[d], p[d] + 1, device="cuda") for d in (2, 1, 0)])
        j = [c[d][:, None] + off[None, :, 2 - d] for d in range(3)]
        there = torch.ones_like(j[0], dtype=torch.bool)
        for d in range(3):
            there &= (j[d] >= 0) & (j[d] < nc[d])
        nbr = torch.where(there, j[0] + nc[0] * (j[1] + nc[1] * j[2]), torch.zeros_like(j[0]))
        nd = off.shape[0]
        A = torch.zeros(self.ncp * nd, 9, dtype=torch.float64, device="cuda")
        for el in self.chunks(4 * (3 * self.n) ** 2):
            K = self.stiffness(el).permute(0, 1, 3, 2, 4).reshape(-1, 9)
            ien = self.ien[el]
            a, b = ien[:, :, None], ien[:, None, :]
            slot = 0
            for d, s in ((2, nc[0] * nc[1]), (1, nc[0]), (0, 1)):
                slot = slot * (2 * p[d] + 1) + (b // s % nc[d] - a // s % nc[d] + p[d])
            A.index_add_(0, (a * nd + slot).reshape(-1), K)
        return A.reshape(self.ncp, nd, 3, 3).transpose(1, 2).contiguous(), nbr, there

    def solve(self, F, rtol=1e-13, most=20000):
        """K u = F with the face x = 0 held, by conjugate gradients on the assembled blocks."""
        A, nbr, _ = self.assembled()
        diag = A[:, :, nbr.shape[1] // 2, :].diagonal(dim1=1, dim2=2).contiguous()
        A = A.reshape(self.ncp, 3, -1)
        free = (torch.arange(self.ncp, device="cuda") % self.nc[0] > 0).double()[:, None]
        r = F.reshape(-1, 3) * free
        x, z = torch.zeros_like(r), r / diag
        q, rz, stop = z.clone(), (r * z).sum(), rtol * r.norm().item()
        for it in range(most):
            y = torch.bmm(A, q[nbr].reshape(self.ncp, -1, 1))[..., 0] * free
            a = rz / (q * y).sum()
            x, r = x + a * q, r - a * y
            if it % 50 == 49 and r.norm().item() <= stop:
                break
            z = r / diag
            new = (r * z).sum()
            q, rz = z + new / rz * q, new
        return x.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        out = []
        for r in _requests(case, seed):
            if r.nb_cp * (2 * r.p + 1) ** 3 > 1500000:
                out.append(None)   # the plain solve of the larger ones takes too long
                continue
            a = r.model()
            c = _case("solve", r.nel, r.p)
            nc = [r.nel[d] + r.p for d in range(3)]
            w = np.empty(r.nb_cp)
            w[_connectivity(r.nel, (r.p,) * 3, nc).ravel()] = a["weight"]
            q = _Exact(c, a["COORDS3D"], w, E=r.E, nu=r.nu)
            out.append(q.solve(q.load(r.traction)))
        return out if any(x is not None for x in out) else None
    nel, p, _ = _dims(case)
    X, w, _ = _net(nel, p, seed)
    if kind == "reassemble":
        X, _, _ = _net(nel, p, seed + 1)
    q = _Exact(case, X, w)
    if kind == "assemble":
        return [q.packed(q.stiffness), None, None, q.load(TRACTION)]
    if kind == "reassemble":
        return [q.packed(q.stiffness), q.load(TRACTION)]
    if kind == "mass":
        return [q.packed(q.mass), None, None]
    if kind == "csr":
        A, _, there = q.assembled()
        y = q.product(_fields(case, seed, 1)[0])
        return [A[there[:, None, :].expand(-1, 3, -1)].reshape(-1), y]
    if kind == "apply":
        g = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.randn(3 * q.ncp, generator=g, device="cuda", dtype=torch.float64)
        return q.product(x.float().double() if case["bits"] == 32 else x)
    if kind == "vib":
        f = _fields(case, seed, case["modes"])
        g, m = q.forms([(u, u, lam) for u, lam in zip(f, np.linspace(1e6, 4e7, case["modes"]))])
        return torch.stack([a.T / b for a, b in zip(g, m)])
    if kind == "shape":
        f = _fields(case, seed, 1 + case["adjoints"])
        g, _ = q.forms([(f[0], v, 0.0) for v in f[1:]])
        vol, gvol = q.volume()
        return [torch.stack([-a.reshape(-1) for a in g]), torch.zeros(case["adjoints"], 3 * q.ncp, dtype=torch.float64),
                vol, gvol]
    # compliance: dJ/dX = -u (dK/dX) u + 2 u (dF/dX), the second by differentiating the load
    F = q.load(TRACTION)
    u = q.solve(F)
    g, _ = q.forms([(u, u, 0.0)])
    q.X = q.X.clone().requires_grad_(True)
    (du,) = torch.autograd.grad(2.0 * torch.dot(q.load(TRACTION), u), q.X)
    return [torch.dot(F, u), (du - g[0]).reshape(-1)]
