"""Performance cases of the femeko_hip library: what a magnetostatics program
has it do, through the package's public entry points, from the smallest mesh
of the tests to the 4.2M-node workload of bench.py.

Meshes are the jittered Kuhn boxes of the repository's workloads ([-1, 1]^3,
n cells per side, six tetrahedra per cell), built here with torch so that a
case is set up quickly. ``scattered`` meshes carry the same geometry in the
numbering of a mesh generator: nodes and elements in random order.

A state of ``prepare`` holds what a user's program keeps between calls: the
host MESH with its device copy, host arrays of coefficients and boundary
data. Relative tolerances are those of the repository's configurations
(1e-10; 1e-12 for gradients), one decade tighter for the FP32-refined solves,
whose potential is further from the solution at the same residual.

``exact`` computes the same quantities with plain torch in 64 bits (assembly
by sorting element entries, CG far below the caller's tolerance).
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "femeko.jl_amd"))

import femeko_hip as fk  # noqa: E402
from femeko_hip.adjoint import fieldObjectiveGradient  # noqa: E402
from femeko_hip.batch import Batch  # noqa: E402

MU0 = math.pi * 4e-7
DEV = "cuda"


# --------------------------------------------------------------------------
# the cases

def listed():
    return [
        # the smallest real call: one linear Dirichlet problem of the tests'
        # size (9,261 nodes), assembled, solved and turned into H, in the
        # reference's precision; launches and latency count
        {"name": "linear20", "kind": "linear", "n": 20, "precision": "f64", "scattered": False},
        # the same at an odd size in the mixed-precision option
        {"name": "linear33-f32", "kind": "linear", "n": 33, "precision": "f32", "scattered": False},
        # an ordinary FP64 model of a quarter million nodes
        {"name": "linear63-f64", "kind": "linear", "n": 63, "precision": "f64", "scattered": False},
        # an ordinary model from a mesh generator: no stencil numbering, so
        # the library renumbers and streams its general matrix copy
        {"name": "scattered55-f32", "kind": "linear", "n": 55, "precision": "f32", "scattered": True},
        # the headline size (4.2M nodes): assembly and FP32-refined solve on
        # resident coefficients, potential, |H| and energy read back
        {"name": "boxes160-f32", "kind": "boxes", "n": 160, "precision": "f32"},
        # the reference's own driver: Neumann load and Lagrange multiplier,
        # on a generator's numbering, FP64
        {"name": "saddle41", "kind": "saddle", "n": 41, "precision": "f64", "scattered": True},
        # the nonlinear workload: Picard/Newton with the Froehlich law, 1.03M
        # nodes, FP64 update solves
        {"name": "froehlich100", "kind": "froehlich", "n": 100, "precision": "f64"},
        # many uneven small meshes, three applied fields each
        {"name": "batch20", "kind": "batch", "count": 20, "nmin": 10, "nmax": 40},
        # design gradient: state and adjoint solve, gradient for every element
        {"name": "adjoint80", "kind": "adjoint", "n": 80, "precision": "f64"},
        # one demagnetizing field of a time-stepping loop on a resident matrix
        {"name": "demag50", "kind": "demag", "n": 50, "precision": "f64"},
        # the sparse matrix itself, handed to the caller's own solver
        {"name": "stiffness60", "kind": "stiffness", "n": 60, "scattered": False},
        # the reference's native bridge: mesh upload, pattern, assembly and
        # singular solve in one stateless call
        {"name": "bridge27", "kind": "bridge", "n": 27, "scattered": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "boxes", "saddle", "froehlich", "batch", "adjoint", "demag", "stiffness",
                       "bridge"])
    prec = rng.choice(["f64", "f32"])
    scat = rng.random() < 0.4
    if kind == "linear":
        return {"kind": kind, "n": _log_int(rng, 9, 72), "precision": prec, "scattered": scat}
    if kind == "boxes":
        return {"kind": kind, "n": _log_int(rng, 70, 140), "precision": prec}
    if kind == "saddle":
        return {"kind": kind, "n": _log_int(rng, 12, 56), "precision": prec, "scattered": scat}
    if kind == "froehlich":
        return {"kind": kind, "n": _log_int(rng, 16, 90), "precision": prec}
    if kind == "batch":
        lo = rng.randint(6, 14)
        return {"kind": kind, "count": _log_int(rng, 3, 40), "nmin": lo, "nmax": lo + rng.randint(4, 30)}
    if kind == "adjoint":
        return {"kind": kind, "n": _log_int(rng, 16, 80), "precision": prec}
    if kind == "demag":
        return {"kind": kind, "n": _log_int(rng, 14, 64), "precision": prec}
    if kind == "stiffness":
        return {"kind": kind, "n": _log_int(rng, 12, 72), "scattered": scat}
    return {"kind": kind, "n": _log_int(rng, 8, 36), "scattered": scat}


# --------------------------------------------------------------------------
# inputs, from the seed alone

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 12345)
    return g


def _rand(gen, *shape):
    return torch.rand(*shape, generator=gen, device=DEV, dtype=torch.float64)


_OFFS = []
for _a, _b, _odd in ((0, 1, 0), (0, 2, 1), (1, 0, 1), (1, 2, 0), (2, 0, 0), (2, 1, 1)):
    _v1 = [0, 0, 0]
    _v1[_a] = 1
    _v2 = list(_v1)
    _v2[_b] = 1
    _q = [[0, 0, 0], _v1, _v2, [1, 1, 1]]
    if _odd:
        _q[2], _q[3] = _q[3], _q[2]
    _OFFS.append(_q)


def _grid(n, jitter, gen, scattered=False):
    """Nodes (nv, 3), 0-based elements (nt, 4) and the box-face node mask on the GPU."""
    m = n + 1
    i = torch.arange(m, device=DEV)
    K, J, I = (v.reshape(-1) for v in torch.meshgrid(i, i, i, indexing="ij"))
    h = 2.0 / n
    idx = torch.stack([I, J, K], 1)
    p = -1.0 + idx.double() * h
    face = ((idx == 0) | (idx == n)).any(1)
    p[face.logical_not()] += ((2.0 * _rand(gen, m ** 3, 3) - 1.0) * (jitter * h))[face.logical_not()]
    p[idx == n] = 1.0
    c = torch.arange(n, device=DEV)
    ck, cj, ci = (v.reshape(-1) for v in torch.meshgrid(c, c, c, indexing="ij"))
    base = ci + m * (cj + m * ck)
    off = torch.tensor([[q[0] + m * (q[1] + m * q[2]) for q in tet] for tet in _OFFS], device=DEV)
    t = (base[:, None, None] + off[None]).reshape(-1, 4)
    if scattered:
        perm = torch.randperm(m ** 3, generator=gen, device=DEV)
        inv = torch.empty_like(perm)
        inv[perm] = torch.arange(m ** 3, device=DEV)
        p, face, t = p[perm], face[perm], inv[t]
        t = t[torch.randperm(t.shape[0], generator=gen, device=DEV)]
    return p, t, face


def _in_box(p, t, lo, hi):
    c = p[t].mean(1)
    lo = torch.as_tensor(lo, device=DEV, dtype=torch.float64)
    hi = torch.as_tensor(hi, device=DEV, dtype=torch.float64)
    return ((c >= lo) & (c <= hi)).all(1)


def _surface(p, t):
    """Outer faces (ns, 3) with outward unit normals and areas."""
    nv = p.shape[0]
    loc = torch.tensor([[1, 2, 3], [0, 2, 3], [0, 1, 3], [0, 1, 2]], device=DEV)
    f = t[:, loc].reshape(-1, 3)
    opp = t.reshape(-1)
    s = f.sort(1).values
    _, inv, cnt = torch.unique((s[:, 0] * nv + s[:, 1]) * nv + s[:, 2], return_inverse=True, return_counts=True)
    outer = cnt[inv] == 1
    f, opp = f[outer], opp[outer]
    nr = torch.linalg.cross(p[f[:, 1]] - p[f[:, 0]], p[f[:, 2]] - p[f[:, 0]])
    a2 = nr.norm(dim=1)
    nr = nr / a2[:, None]
    flip = (nr * (p[opp] - p[f[:, 0]])).sum(1) > 0
    nr[flip] *= -1
    return f, nr, a2 / 2


def _batch_sizes(case):
    """Cells per side of a batch's meshes: nmin..nmax in golden-ratio steps."""
    span = case["nmax"] - case["nmin"] + 1
    return [case["nmin"] + int(((k + 0.5) * 0.6180339887498949 % 1.0) * span) for k in range(case["count"])]


def _inputs(case, seed):
    """Everything a case is made of, as GPU tensors."""
    gen, kind = _gen(seed), case["kind"]
    if kind == "batch":
        out = []
        for n in _batch_sizes(case):
            p, t, face = _grid(n, 0.2, gen)
            c, s = (-0.7 + 1.4 * _rand(gen, 3)), (0.1 + 0.5 * _rand(gen, 3))
            mur = 10.0 + 990.0 * _rand(gen, 1)
            mu = MU0 * torch.where(_in_box(p, t, c - s / 2, c + s / 2), mur, torch.ones_like(mur))
            out.append({"p": p, "t": t, "face": face, "mu": mu, "g": [torch.where(face, -p[:, k], 0.0)
                                                                     for k in range(3)]})
        return out
    p, t, face = _grid(case["n"], 0.15 if kind == "boxes" else 0.2, gen, case.get("scattered", False))
    d = {"p": p, "t": t, "face": face}
    nt = t.shape[0]
    magnet = _in_box(p, t, [-0.25] * 3, [0.25] * 3)
    d["magnet"] = magnet
    if kind in ("linear", "saddle", "bridge"):
        mur = 100.0 + 1900.0 * _rand(gen, 1)
        d["mu"] = MU0 * torch.where(magnet, mur, torch.ones_like(mur))
    elif kind == "boxes":
        inside = torch.zeros(nt, dtype=torch.bool, device=DEV)
        for _ in range(8):
            c, s = (-0.7 + 1.4 * _rand(gen, 3)), (0.1 + 0.5 * _rand(gen, 3))
            inside |= _in_box(p, t, c - s / 2, c + s / 2)
        d["mu"] = MU0 * torch.where(inside, 10.0 ** (3.0 * _rand(gen, nt)), 1.0)
    elif kind == "froehlich":
        d["mu"] = torch.full((nt,), MU0, device=DEV, dtype=torch.float64)
    elif kind == "adjoint":
        d["rho"] = _rand(gen, nt)
        d["mu"] = MU0 * (1.0 + 999.0 * d["rho"] ** 3)
        d["target"] = _in_box(p, t, [-0.2] * 3, [0.2] * 3)
    elif kind == "demag":
        a = 6.0 * _rand(gen, 3)
        w = torch.stack([torch.sin(a[0] * p[:, 1] + a[1]), torch.cos(a[0] * p[:, 0]), torch.sin(a[2] * p[:, 2])], 1)
        w = w + 0.2 * (_rand(gen, p.shape[0], 3) - 0.5)
        on = torch.zeros(p.shape[0], dtype=torch.bool, device=DEV)
        on[t[magnet].reshape(-1)] = True
        d["M"] = 8e5 * torch.where(on[:, None], w / w.norm(dim=1, keepdim=True), 0.0)
    elif kind == "stiffness":
        d["mu"] = MU0 * (1.0 + 999.0 * _rand(gen, nt))
    H0 = torch.tensor([1.0, 0.0, 0.0], device=DEV, dtype=torch.float64)
    if kind == "froehlich":
        H0 = 2.0 * _rand(gen, 3) - 1.0
        H0 = 1e4 * H0 / H0.norm()
    d["H0"] = H0
    d["g"] = torch.where(face, -(p @ H0), 0.0)
    if kind in ("saddle", "bridge"):
        d["surface"] = _surface(p, t)
    return d


def _host_mesh(d):
    p, t = d["p"], d["t"]
    mesh = fk.MESH(p=p.cpu().numpy().T, t=(t + 1).to(torch.int32).cpu().numpy().T, VE=_volumes(p, t).cpu().numpy())
    if "surface" in d:
        f, nr, ae = d["surface"]
        sT = torch.ones(f.shape[0], 4, dtype=torch.int32, device=DEV)
        sT[:, :3] = f + 1
        mesh.surfaceT, mesh.normal, mesh.AE = sT.cpu().numpy().T, nr.cpu().numpy().T, ae.cpu().numpy()
        mesh.shell_id = (1,)
    return mesh


def _np(x):
    return x.cpu().numpy()


def _rtol(case):
    return 1e-12 if case["kind"] == "adjoint" else 1e-11 if case.get("precision") == "f32" else 1e-10


def prepare(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    s = {"case": case, "rtol": _rtol(case)}
    if kind == "batch":
        meshes = [_host_mesh(x) for x in d]
        s["batch"] = Batch(meshes, nrhs=3)
        s["mus"] = [_np(x["mu"]) for x in d]
        s["batch"].set_dirichlet([_np(x["face"]) for x in d], [_np(torch.stack(x["g"])) for x in d])
        return s
    s["mesh"] = mesh = _host_mesh(d)
    if "mu" in d:
        s["mu"] = _np(d["mu"])
    if kind == "bridge":
        s["H0"] = _np(MU0 * d["H0"])
        return s
    dm = fk.device_mesh(mesh)
    s["mask"], s["g"] = _np(d["face"]).astype(np.uint8), _np(d["g"])
    if kind == "boxes":
        dm.set_coefficient(s["mu"])
        dm.set_dirichlet(s["mask"], s["g"])
    elif kind == "saddle":
        s["H0"] = _np(MU0 * d["H0"])
    elif kind == "froehlich":
        s["region"] = _np(d["magnet"]).astype(np.uint8)
        dm.set_dirichlet(s["mask"], s["g"])
        dm.set_inner_precision(case["precision"])
    elif kind == "adjoint":
        s["rho"], s["target"] = _np(d["rho"]), _np(d["target"]).astype(np.uint8)
    elif kind == "demag":
        s["inside"] = _np(d["magnet"]).astype(np.uint8)
        s["M"] = _np(d["M"]).T
        s["volumes"] = _np(_node_volumes(d))
        dm.set_coefficient(np.ones(mesh.nt))
        dm.assemble()
        dm.set_inner_precision(case["precision"])
    return s


# --------------------------------------------------------------------------
# one pass

def run(s):
    case, mesh = s["case"], s.get("mesh")
    kind = case["kind"]
    if kind == "linear":
        u, _rep = fk.solveDirichlet(mesh, s["mu"], s["mask"], s["g"], rtol=s["rtol"], precision=case["precision"])
        return {"u": u, "H": fk.magneticField(mesh, u)}
    if kind == "boxes":
        dm = fk.device_mesh(mesh)
        dm.assemble()
        dm.solve(case["precision"], rtol=s["rtol"])
        u = dm.potential()
        _H, Hn, E = dm.field(want_H=False, want_energy=True)
        return {"u": u, "Hn": Hn, "energy": np.float64(E)}
    if kind == "saddle":
        b = -fk.BoundaryIntegral(mesh, s["H0"], mesh.shell_id)
        u, _mult = fk.solveSaddle(mesh, s["mu"], b, s["rtol"], case["precision"])
        return {"u": u, "H": fk.magneticField(mesh, u)}
    if kind == "froehlich":
        dm = fk.device_mesh(mesh)
        dm.nonlinear_froehlich(s["region"], 1.2e6, 500.0, rtol=s["rtol"], tol_mu=1e-6, max_outer=20)
        return {"u": dm.potential(), "mu": dm.get_coefficient()}
    if kind == "batch":
        b = s["batch"]
        b.set_coefficient(s["mus"])
        b.assemble()
        b.solve(rtol=1e-11)
        return [b.potential(m) for m in range(b.nmesh)]
    if kind == "adjoint":
        J, grad, _it = fieldObjectiveGradient(mesh, s["rho"], s["target"], (2.0, 0.0, 0.0), s["mask"], s["g"],
                                              rtol=s["rtol"], precision=case["precision"])
        return {"J": np.float64(J), "grad": grad}
    if kind == "demag":
        Hd, _it, _rel = fk.device_mesh(mesh).demag_field(s["inside"], s["M"], s["volumes"], rtol=s["rtol"])
        return Hd
    if kind == "stiffness":
        A = fk.stiffnessMatrix(mesh, s["mu"])
        return {"colptr": A.indptr, "rowval": A.indices, "nzval": A.data}
    return fk.scalarPotential(mesh, s["mu"], s["H0"], mesh.shell_id[0])


# --------------------------------------------------------------------------
# what one pass cannot do without

def _sizes(n):
    m = n + 1
    return m ** 3, 6 * n ** 3, m ** 3 + 2 * (3 * n * m * m + 3 * n * n * m + n ** 3)


def work(case):
    """Bytes: each host input read and each output written once. Operations:
    assembly (about 170 per element for gradients and the ten distinct
    entries) and, per Jacobi-PCG iteration, 2 per stored entry and 11 per
    node; iterations grow with n (about 8 n per solve to 1e-10 here)."""
    kind = case["kind"]
    if kind == "batch":
        w = {"bytes": 0.0, "flops": 0.0}
        for n in _batch_sizes(case):
            nv, nt, nnz = _sizes(n)
            w["bytes"] += 8 * nt + 24 * nv
            w["flops"] += 170 * nt + 3 * 8 * n * (2 * nnz + 11 * nv)
        return w
    n = case["n"]
    nv, nt, nnz = _sizes(n)
    cg = 8 * n * (2 * nnz + 11 * nv)
    asm = 170 * nt
    if kind == "linear":
        return {"bytes": 32 * nt + 17 * nv, "flops": asm + cg + 30 * nt}
    if kind == "boxes":
        return {"bytes": 16 * nt + 8 * nv, "flops": asm + cg + 30 * nt}
    if kind == "saddle":
        return {"bytes": 32 * nt + 16 * nv, "flops": asm + cg + 30 * nt}
    if kind == "froehlich":
        return {"bytes": 9 * nt + 8 * nv, "flops": 8 * (2 * asm + 0.7 * cg)}
    if kind == "adjoint":
        return {"bytes": 17 * nt + 9 * nv, "flops": asm + 2 * cg + 60 * nt}
    if kind == "demag":
        return {"bytes": nt + 56 * nv, "flops": cg + 30 * nt}
    if kind == "stiffness":
        return {"bytes": 8 * nt + 12 * nnz + 4 * nv, "flops": asm}
    return {"bytes": 16 * nt + 24 * nv + 16 * nt + 8 * nv, "flops": asm + cg}


# --------------------------------------------------------------------------
# the same in 64 bits with plain torch

def _gradients(p, t):
    """(nt, 4, 3) basis gradients and (nt,) volumes."""
    e = p[t[:, 1:]] - p[t[:, :1]]
    a, b, c = e[:, 0], e[:, 1], e[:, 2]
    bc = torch.linalg.cross(b, c)
    det = (a * bc).sum(1)
    g = torch.stack([bc, torch.linalg.cross(c, a), torch.linalg.cross(a, b)], 1) / det[:, None, None]
    return torch.cat([-g.sum(1, keepdim=True), g], 1), det.abs() / 6.0


def _volumes(p, t):
    e = p[t[:, 1:]] - p[t[:, :1]]
    return (e[:, 0] * torch.linalg.cross(e[:, 1], e[:, 2])).sum(1).abs() / 6.0


def _node_volumes(d):
    t = d["t"][d["magnet"]]
    v = torch.zeros(d["p"].shape[0], device=DEV, dtype=torch.float64)
    return v.index_add_(0, t.reshape(-1), _volumes(d["p"], t).repeat_interleave(4))


class _Pattern:
    """Sorted node pairs of the elements, and the pair of every element entry."""

    def __init__(self, t, nv):
        self.nv = nv
        key, self.slot = torch.unique((t[:, :, None] * nv + t[:, None, :]).reshape(-1), return_inverse=True)
        self.row, self.col = key // nv, key % nv
        self.crow = torch.zeros(nv + 1, dtype=torch.int64, device=DEV)
        self.crow[1:] = torch.bincount(self.row, minlength=nv).cumsum(0)

    def values(self, local):
        v = torch.zeros(self.row.numel(), device=DEV, dtype=torch.float64)
        return v.index_add_(0, self.slot, local.reshape(-1))

    def matrix(self, val):
        return torch.sparse_csr_tensor(self.crow, self.col, val, (self.nv, self.nv))

    def diag(self, val):
        on = self.row == self.col
        d = torch.zeros(self.nv, device=DEV, dtype=torch.float64)
        d[self.row[on]] = val[on]
        return d


def _cg(A, diag, b, free=None, tol=1e-14):
    """Jacobi-CG on the free rows; free=None: the consistent singular system."""
    live = torch.ones_like(b) if free is None else free.double()
    inv = torch.where((live > 0) & (diag > 0), 1.0 / diag, 0.0)
    x, r = torch.zeros_like(b), b * live
    if free is None:
        r = r - r.mean()
    z = inv * r
    q, rz, ref = z.clone(), r @ z, float(r.norm())
    for k in range(20000):
        Aq = (A @ q) * live
        al = rz / (q @ Aq)
        x += al * q
        r -= al * Aq
        if k % 20 == 19 and float(r.norm()) <= tol * ref:
            break
        z = inv * r
        new = r @ z
        q = z + (new / rz) * q
        rz = new
    return x


def _element_field(u, t, G):
    return -(u[t][:, :, None] * G).sum(1)


def _nonlinear(d, pat, G, VE, free):
    Ms, a = 1.2e6, 500.0
    t, u = d["t"], d["g"].clone()
    mu = d["mu"].clone()
    hit, last = None, 1.0
    for k in range(60):
        K = G @ G.transpose(1, 2)
        val = pat.values((VE * mu)[:, None, None] * K)
        res = -(pat.matrix(val) @ u)
        if last < 0.25:
            gh = (G * hit[:, None, :]).sum(2)
            hn = hit.norm(dim=1)
            dmu = torch.where(d["magnet"], -MU0 * Ms / (a + hn) ** 2, 0.0)
            val = val + pat.values((VE * dmu / hn.clamp_min(1e-300))[:, None, None] * gh[:, :, None] * gh[:, None, :])
        u = u + _cg(pat.matrix(val), pat.diag(val), res, free, 1e-13 if last > 1e-3 else 1e-8)
        hit = _element_field(u, t, G)
        new = torch.where(d["magnet"], MU0 * (1.0 + Ms / (a + hit.norm(dim=1))), MU0)
        last = float(((new - mu).abs() / new).max())
        mu = new
        if last < 1e-12:
            break
    return {"u": u, "mu": mu}


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    if kind == "batch":
        at, parts = 0, []
        for x in d:
            parts.append(x["t"] + at)
            at += x["p"].shape[0]
        p, t = torch.cat([x["p"] for x in d]), torch.cat(parts)
        free = torch.cat([x["face"] for x in d]).logical_not()
        G, VE = _gradients(p, t)
        pat = _Pattern(t, at)
        val = pat.values((VE * torch.cat([x["mu"] for x in d]))[:, None, None] * (G @ G.transpose(1, 2)))
        A, dg, us = pat.matrix(val), pat.diag(val), []
        for k in range(3):
            g = torch.cat([x["g"][k] for x in d])
            us.append(g + _cg(A, dg, -(A @ g), free))
        u, out, at = torch.stack(us), [], 0
        for x in d:
            out.append(u[:, at:at + x["p"].shape[0]].contiguous())
            at += x["p"].shape[0]
        return out
    p, t, face = d["p"], d["t"], d["face"]
    free = face.logical_not()
    G, VE = _gradients(p, t)
    pat = _Pattern(t, p.shape[0])
    if kind == "froehlich":
        return _nonlinear(d, pat, G, VE, free)
    mu = d["mu"] if "mu" in d else torch.ones(t.shape[0], device=DEV, dtype=torch.float64)
    val = torch.zeros(pat.row.numel(), device=DEV, dtype=torch.float64)
    for i in range(4):  # one row of the element matrices at a time: the largest mesh has 393M entries
        loc = (VE * mu)[:, None] * (G[:, i:i + 1] * G).sum(2)
        val.index_add_(0, pat.slot.reshape(-1, 4, 4)[:, i].reshape(-1), loc.reshape(-1))
    if kind == "stiffness":
        return {"colptr": None, "rowval": None, "nzval": val}
    A, dg = pat.matrix(val), pat.diag(val)
    lag = torch.zeros(p.shape[0], device=DEV, dtype=torch.float64)
    lag.index_add_(0, t.reshape(-1), (VE / 4).repeat_interleave(4))
    if kind in ("linear", "boxes"):
        u = d["g"] + _cg(A, dg, -(A @ d["g"]), free)
        H = _element_field(u, t, G)
        if kind == "linear":
            return {"u": u, "H": H.T}
        return {"u": u, "Hn": H.norm(dim=1), "energy": 0.5 * (mu * VE * (H * H).sum(1)).sum()}
    if kind in ("saddle", "bridge"):
        f, nr, ae = d["surface"]
        b = torch.zeros(p.shape[0], device=DEV, dtype=torch.float64)
        b.index_add_(0, f.reshape(-1), ((nr @ (MU0 * d["H0"])) * ae / 3).repeat_interleave(3))
        u = _cg(A, dg, -b)
        if kind == "bridge":
            return u - (dg @ u) / dg.sum()
        u = u - (lag @ u) / lag.sum()
        return {"u": u, "H": _element_field(u, t, G).T}
    if kind == "adjoint":
        u = d["g"] + _cg(A, dg, -(A @ d["g"]), free)
        H, tg = _element_field(u, t, G), d["target"]
        diff = torch.where(tg[:, None], H - torch.tensor([2.0, 0.0, 0.0], device=DEV, dtype=torch.float64), 0.0)
        dJ = torch.zeros_like(u)
        dJ.index_add_(0, t.reshape(-1), (-2.0 * VE[:, None] * (G * diff[:, None, :]).sum(2)).reshape(-1))
        lam = _cg(A, dg, -dJ, free)
        grad = VE * (_element_field(lam, t, G) * H).sum(1) * MU0 * 2997.0 * d["rho"] ** 2
        return {"J": (VE[:, None] * diff * diff).sum(), "grad": grad}
    M, inside = d["M"], d["magnet"]
    ti = t[inside]
    load = VE[inside, None] * (G[inside] * M[ti].mean(1)[:, None, :]).sum(2)
    b = torch.zeros(p.shape[0], device=DEV, dtype=torch.float64).index_add_(0, ti.reshape(-1), load.reshape(-1))
    u = _cg(A, dg, b)
    h = VE[inside, None] * _element_field(u, ti, G[inside])
    Hd = torch.zeros_like(p).index_add_(0, ti.reshape(-1), h.repeat_interleave(4, 0))
    return (Hd / _node_volumes(d)[:, None]).T
