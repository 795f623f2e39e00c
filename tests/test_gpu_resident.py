"""The register-resident PCG (one cooperative launch per solve on the stencil
copy) against the three-kernel iteration, which a context with timing enabled
runs: row counts at the edges of its launch shapes, elongated grids whose
windows merge or split, odd tails, iteration limit and breakdown.

Bars: both solves stop at ||r|| < 1e-12 ||b||, so their potentials agree to
the suite's 1e-9; FP64 iteration counts agree to 5% + 4 (rounding moves the
iteration at which a slowly falling residual crosses the tolerance; the FP32
recursions' counts depend on when each is replaced and are not compared)."""
import numpy as np
import pytest

from femeko_hip import FemekoHIPError
from femeko_hip import workloads as W
from femeko_hip.device import Context, DeviceMesh
from femeko_hip.mesh import MESH, MU0, _kuhn_local_offsets, element_volumes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def contexts():
    plain, timed = Context(0), Context(0)
    timed.set_timing(True)
    yield plain, timed
    plain.close()
    timed.close()


def _box(nx, ny, nz):
    """Kuhn mesh of nx x ny x nz unit cells, x fastest."""
    m, l = nx + 1, ny + 1
    K, J, I = np.meshgrid(np.arange(nz + 1), np.arange(l), np.arange(m), indexing="ij")
    p = np.asfortranarray(np.stack([I.ravel(), J.ravel(), K.ravel()]).astype(float))
    ck, cj, ci = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    base = (ci + m * (cj + l * ck)).ravel()
    off = _kuhn_local_offsets()
    t = base[:, None, None] + (off[:, :, 0] + m * (off[:, :, 1] + l * off[:, :, 2]))[None]
    t = np.asfortranarray((t.reshape(-1, 4).T + 1).astype(np.int32))
    return MESH(p=p, t=t, VE=element_volumes(p, t))


def _both(contexts, mesh, mu, mask, g, precision="f64", rtol=1e-12, fmt=None):
    out = []
    for ctx in contexts:
        dm = DeviceMesh(mesh, ctx)
        try:
            dm.set_coefficient(mu)
            dm.assemble()
            dm.set_dirichlet(mask, g)
            rep = dm.solve(precision, rtol=rtol)
            assert fmt is None or dm.solver_format()[0] == fmt
            first = dm.potential()
            again = dm.solve(precision, rtol=rtol)
            assert np.array_equal(first, dm.potential()) and again.iterations == rep.iterations
            out.append((first, rep))
        finally:
            dm.close()
    (a, ra), (b, rb) = out
    assert ra.relres < rtol and rb.relres < rtol
    assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
    if precision == "f64":
        assert abs(ra.iterations - rb.iterations) <= 4 + rb.iterations // 20


def _increment(contexts, n, precision):
    """The composite solves that run the FP32 recursion on a right-hand side
    of their own (adjoint) and on every row (Neumann)."""
    pr = W.adjoint(n)
    rng = np.random.default_rng(n)
    b = rng.normal(size=pr.mesh.nv)
    b -= b.mean()
    out = []
    for ctx in contexts:
        dm = DeviceMesh(pr.mesh, ctx)
        try:
            dm.set_coefficient(pr.mu)
            dm.assemble()
            dm.set_dirichlet(pr.mask, pr.g)
            dm.set_inner_precision(precision)
            dm.solve("f64", rtol=1e-12)
            J, grad, _ = dm.adjoint_field_target(pr.magnet.astype(np.uint8), (2.0, 0.0, 0.0), rtol=1e-12)
            u, _m, _it, rel = dm.solve_neumann(b, rtol=1e-12)
            assert rel < 1e-12
            out.append((J, grad, u))
        finally:
            dm.close()
    (Ja, ga, ua), (Jb, gb, ub) = out
    assert abs(Ja - Jb) <= 1e-9 * abs(Jb)
    assert np.linalg.norm(ga - gb) <= 1e-8 * np.linalg.norm(gb)
    assert np.linalg.norm(ua - ub) <= 1e-8 * np.linalg.norm(ub)


# 27 rows; 512 rows exactly; one more plane; the last n of each launch shape
# and the first of the next (rows (n + 1)^3 against 256 x 512, 1024, ... 4096)
@pytest.mark.parametrize("n", [2, 7, 8, 19, 49, 50, 63, 64, 72, 73, 79, 80, 85, 86, 90, 91, 95, 96, 100, 101])
def test_launch_shapes(contexts, n):
    pr = W.linear(n)
    _both(contexts, pr.mesh, pr.mu, pr.mask, pr.g, fmt="stencil")


@pytest.mark.parametrize("n", [2, 7, 19, 49, 50, 63, 64, 79, 80, 90, 91, 100, 101, 115, 116, 126, 127])
def test_launch_shapes_f32(contexts, n):
    pr = W.linear(n)
    _both(contexts, pr.mesh, pr.mu, pr.mask, pr.g, precision="f32", fmt="stencil")


# bricks: the last n of a shape and the first of the next, up to the last mesh
# that fits (FP64 n = 131, FP32 n = 162) and one past it (three kernels)
@pytest.mark.parametrize("precision,n", [("f64", n) for n in (83, 84, 95, 102, 103, 107, 113, 119, 127, 130)]
                         + [("f32", n) for n in (83, 87, 102, 118, 130, 134, 143, 151, 162, 163)])
def test_brick_shapes(contexts, precision, n):
    pr = W.linear(n)
    _both(contexts, pr.mesh, pr.mu, pr.mask, pr.g, precision=precision, fmt="stencil")


# bricks of grids that are no cubes: two runs per plane over 120 layers; one
# layer of few planes; short last runs and last layers
@pytest.mark.parametrize("dims", [(30, 30, 600), (400, 400, 3), (230, 47, 55), (61, 201, 43), (90, 13, 500)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_brick_grids(contexts, dims, precision):
    mesh = _box(*dims)
    rng = np.random.default_rng(5)
    mu = MU0 * rng.uniform(1.0, 50.0, mesh.nt)
    mask = ((mesh.p == 0.0) | (mesh.p == np.array(dims, float)[:, None])).any(axis=0)
    g = np.where(mask, rng.normal(size=mesh.nv), 0.0)
    _both(contexts, mesh, mu, mask.astype(np.uint8), g, precision=precision)


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n", [12, 34, 84])
def test_right_hand_sides(contexts, n, precision):
    _increment(contexts, n, precision)


# a mesh generator's numbering: the SELL copy of the renumbered mesh, at the
# edges of its launch shapes (512, 1024, 1536, 2048 rows per block)
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n", [3, 8, 20, 49, 50, 63, 64, 72, 73, 79, 80])
def test_scattered_numbering(contexts, n, precision):
    pr = W.linear(n)
    pr = W.renumbered(pr, np.random.default_rng(n).permutation(pr.mesh.nv), "scattered")
    order = np.random.default_rng(n + 1).permutation(pr.mesh.nt)
    mesh = MESH(p=pr.mesh.p, t=np.asfortranarray(pr.mesh.t[:, order]), VE=pr.mesh.VE[order])
    _both(contexts, mesh, pr.mu[order], pr.mask, pr.g, precision=precision)


# Delaunay meshes: rows of 4 to over 30 entries (beyond 32: the three kernels)
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("points", [60, 700, 9000])
def test_delaunay(contexts, points, precision):
    from scipy.spatial import Delaunay

    rng = np.random.default_rng(points)
    pts = np.concatenate([rng.random((points, 3)), np.array([[i, j, k] for i in (0, 1) for j in (0, 1)
                                                             for k in (0, 1)], float)])
    tri = Delaunay(pts, qhull_options="QJ").simplices
    p = np.asfortranarray(pts.T)
    t = np.asfortranarray((tri.T + 1).astype(np.int32))
    vol = element_volumes(p, t)
    t = np.asfortranarray(t[:, vol > 1e-9])
    mesh = MESH(p=p, t=t, VE=element_volumes(p, t))
    used = np.zeros(mesh.nv, bool)
    used[t.ravel() - 1] = True
    mask = (~used) | (p[2] < 0.15) | (p[2] > 0.85)
    g = np.where(mask, p[2], 0.0)
    mu = MU0 * rng.uniform(1.0, 20.0, mesh.nt)
    _both(contexts, mesh, mu, mask.astype(np.uint8), g, precision=precision)


# one cell thick (too much padding for the stencil copy: SELL), long columns,
# flat plates: one merged window, split windows, and offsets too far apart for
# three windows (the three-kernel iteration on both)
@pytest.mark.parametrize("dims", [(1, 1, 200), (3, 5, 41), (200, 3, 3), (90, 90, 2), (2, 90, 90), (700, 20, 3)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_elongated_grids(contexts, dims, precision):
    mesh = _box(*dims)
    rng = np.random.default_rng(3)
    mu = MU0 * rng.uniform(1.0, 50.0, mesh.nt)
    top = np.array(dims, float)[:, None]
    mask = ((mesh.p == 0.0) | (mesh.p == top)).any(axis=0)
    inner = rng.random(mesh.nv) < 0.5     # a one-cell box has no interior: free half of its nodes
    mask = mask & ~inner if not (~mask).any() else mask
    g = np.where(mask, rng.normal(size=mesh.nv), 0.0)
    _both(contexts, mesh, mu, mask.astype(np.uint8), g, precision=precision)


def test_limit_and_breakdown(contexts):
    pr = W.linear(20)
    dm = DeviceMesh(pr.mesh, contexts[0])
    try:
        dm.set_coefficient(pr.mu)
        dm.assemble()
        dm.set_dirichlet(pr.mask, pr.g)
        rep = dm.solve("f64", rtol=1e-12, max_iter=7, raise_on_error=False)
        assert rep.status == 6 and rep.iterations == 7
        assert dm.solve("f64", rtol=1e-10).relres < 1e-10
        rep = dm.solve("f32", rtol=1e-12, max_iter=7, raise_on_error=False)
        assert rep.status == 6 and rep.iterations == 7
        # zero Dirichlet data: b = 0, nothing to iterate
        dm.set_dirichlet(pr.mask, np.zeros_like(pr.g))
        assert dm.solve("f64", rtol=1e-10).iterations == 0 and not dm.potential().any()
        # indefinite coefficients that keep every diagonal positive break down or diverge with a status
        mu = pr.mu.copy()
        mu[::7] *= -2.0
        dm.set_coefficient(mu)
        dm.assemble()
        dm.set_dirichlet(pr.mask, pr.g)
        with pytest.raises(FemekoHIPError):
            dm.solve("f64", rtol=1e-12, max_iter=300)
    finally:
        dm.close()


def test_two_contexts_in_two_threads():
    import threading

    probs = [W.linear(40), W.linear(56)]
    ref, got, ctxs, dms = [], [[], []], [Context(0), Context(0)], []
    for pr, ctx in zip(probs, ctxs):
        dm = DeviceMesh(pr.mesh, ctx)
        dm.set_coefficient(pr.mu)
        dm.assemble()
        dm.set_dirichlet(pr.mask, pr.g)
        dm.solve("f64", rtol=1e-10)
        ref.append(dm.potential())
        dms.append(dm)

    def work(k):
        for _ in range(6):
            dms[k].solve("f64", rtol=1e-10)
            got[k].append(dms[k].potential())

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(2):
        dms[k].close()
        ctxs[k].close()
        assert len(got[k]) == 6 and all(np.array_equal(ref[k], u) for u in got[k])


# (boxes nx, ny, nz, right-hand sides): one tiny mesh; rows 511, 512 and 513
# wide of a block (7*73 = 511, 8*64, 9*57); one launch of 512, of 1024 rows a
# block; several launches of 2048 with a mesh that ends a block exactly
@pytest.mark.parametrize("boxes,nrhs", [
    ([(1, 1, 1)], 1),
    ([(6, 72, 1), (6, 6, 2), (7, 7, 7), (18, 8, 2), (1, 1, 400)], 4),
    ([(20, 20, 20)] * 3 + [(3, 4, 5)], 2),
    ([(32, 32, 20), (15, 15, 31), (30, 30, 30), (40, 40, 20)], 3),
    ([(28, 28, 28)] * 7 + [(15, 15, 31), (2, 1, 3)], 3),
])
def test_batch(contexts, boxes, nrhs):
    """Every system a group of blocks of its own; a system without a
    right-hand side stays out. Potentials within the suite's 1e-9 of the
    three-kernel batch at rtol 1e-12."""
    from femeko_hip.batch import Batch

    rng = np.random.default_rng(len(boxes) * 10 + nrhs)
    meshes, mus, masks, gs = [], [], [], []
    for b in boxes:
        mesh = _box(*(max(v, 1) for v in b))
        mask = np.zeros(mesh.nv, np.uint8)
        mask[: (b[0] + 1) * 2] = 1
        mask[-1] = 1
        g = np.where(mask, rng.normal(size=(nrhs, mesh.nv)), 0.0)
        meshes.append(mesh)
        mus.append(MU0 * rng.uniform(1.0, 5.0, mesh.nt))
        masks.append(mask)
        gs.append(g)
    if len(boxes) > 1:
        gs[0][-1][:] = 0.0
    out = []
    for ctx in contexts:
        b = Batch(meshes, nrhs=nrhs, ctx=ctx)
        try:
            b.set_coefficient(mus)
            b.assemble()
            b.set_dirichlet(masks, gs)
            rep = b.solve(rtol=1e-12)
            first = [b.potential(k) for k in range(b.nmesh)]
            again = b.solve(rtol=1e-12)
            assert all(np.array_equal(u, b.potential(k)) for k, u in enumerate(first))
            assert np.array_equal(rep.iterations, again.iterations)
            assert rep.relres.max() < 1e-12
            with pytest.raises(FemekoHIPError):
                b.solve(rtol=1e-12, max_iter=1)
            out.append(first)
        finally:
            b.close()
    for u, v in zip(*out):
        for j in range(nrhs):
            assert np.linalg.norm(u[j] - v[j]) <= 1e-9 * np.linalg.norm(v[j])
