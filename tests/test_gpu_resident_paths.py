"""Which launch a solve takes, and what the other one gives: fk_solve_launch at
the edges of every layout and shape (256 CUs), each solve against a context
that runs three kernels per iteration in captured graphs
(FEMEKO_HIP_RESIDENT=0). Both stop at ||r|| < 1e-12 ||b||: potentials agree to
the suite's 1e-9. The three kernels give the same bits in graphs as launched
one by one with timing enabled."""
import os

import numpy as np
import pytest

from femeko_hip import workloads as W
from femeko_hip.batch import Batch
from femeko_hip.device import Context, DeviceMesh
from femeko_hip.mesh import MESH, MU0, element_volumes
from test_gpu_resident import _box

pytestmark = pytest.mark.gpu

KERNELS = ("kernels", 0)


@pytest.fixture(scope="module")
def contexts():
    plain = Context(0)
    saved = os.environ.get("FEMEKO_HIP_RESIDENT")
    os.environ["FEMEKO_HIP_RESIDENT"] = "0"
    try:
        kernels = Context(0)
    finally:
        if saved is None:
            del os.environ["FEMEKO_HIP_RESIDENT"]
        else:
            os.environ["FEMEKO_HIP_RESIDENT"] = saved
    yield plain, kernels
    plain.close()
    kernels.close()


def _solve(ctx, mesh, mu, mask, g, precision, rtol=1e-12):
    dm = DeviceMesh(mesh, ctx)
    try:
        dm.set_coefficient(mu)
        dm.assemble()
        dm.set_dirichlet(mask, g)
        assert dm.solve_launch() == (None, 0, 0)
        rep = dm.solve(precision, rtol=rtol)
        assert rep.relres < rtol
        rows = np.diff(dm.pattern(0)[0]) - 1
        return dm.potential(), rep, dm.solve_launch(), int(rows.max())
    finally:
        dm.close()


def _check(contexts, mesh, mu, mask, g, precision, expect):
    a, _, launch, _ = _solve(contexts[0], mesh, mu, mask, g, precision)
    b, _, other, _ = _solve(contexts[1], mesh, mu, mask, g, precision)
    assert launch[:2] == expect and (launch[2] > 0) == (expect != KERNELS)
    assert other == ("kernels", 0, 0)
    assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)


# the first n of a shape or the last, the last mesh of bricks and one past it
@pytest.mark.parametrize("precision,n,layout,rows", [
    ("f64", 2, "windows", 512), ("f64", 49, "windows", 512), ("f64", 50, "windows", 1024), ("f64", 64, "windows", 1536),
    ("f64", 79, "windows", 2048), ("f64", 80, "bricks", 2560), ("f64", 85, "bricks", 3072), ("f64", 95, "bricks", 3584),
    ("f64", 100, "bricks", 4608), ("f64", 103, "bricks", 5120), ("f64", 113, "bricks", 6144),
    ("f64", 118, "bricks", 7168), ("f64", 130, "bricks", 9216), ("f64", 131, *KERNELS),
    ("f32", 2, "windows", 512), ("f32", 50, "windows", 1024), ("f32", 64, "windows", 1536), ("f32", 79, "windows", 2048),
    ("f32", 80, "bricks", 2560), ("f32", 87, "bricks", 3072), ("f32", 101, "bricks", 4608), ("f32", 116, "bricks", 7168),
    ("f32", 127, "bricks", 8192), ("f32", 143, "bricks", 12288), ("f32", 151, "bricks", 15360),
    ("f32", 160, "bricks", 16896), ("f32", 165, "bricks", 18432), ("f32", 166, *KERNELS)])
def test_boxes(contexts, precision, n, layout, rows):
    pr = W.linear(n)
    _check(contexts, pr.mesh, pr.mu, pr.mask, pr.g, precision, (layout, rows))


# nodes of every line along x numbered backwards: the boxes are cut along
# another diagonal, offsets 1, a - 1, a, P - 1, P, P + a - 1, P + a, no bricks
@pytest.mark.parametrize("precision,n,layout,rows", [
    ("f64", 30, "windows", 512), ("f64", 85, "windows", 2560), ("f64", 86, "windows", 3072),
    ("f64", 91, "windows", 3072), ("f64", 93, "windows", 3584), ("f64", 96, "windows", 3584),
    ("f64", 98, "windows", 4096), ("f64", 100, "windows", 4096), ("f64", 101, *KERNELS),
    ("f32", 80, "windows", 3072), ("f32", 93, "windows", 4096), ("f32", 100, "windows", 4096),
    ("f32", 101, "windows", 6144), ("f32", 115, "windows", 6144), ("f32", 124, "windows", 8192),
    ("f32", 127, "windows", 8192)])
def test_boxes_cut_the_other_way(contexts, precision, n, layout, rows):
    pr = W.linear(n)
    order = np.arange(pr.mesh.nv).reshape(-1, n + 1)[:, ::-1].ravel()
    pr = W.renumbered(pr, order, "backwards")
    _check(contexts, pr.mesh, pr.mu, pr.mask, pr.g, precision, (layout, rows))


@pytest.mark.parametrize("precision,n,layout,rows", [
    ("f64", 20, "sell", 512), ("f64", 50, "sell", 1024), ("f64", 72, "sell", 1536), ("f64", 73, *KERNELS),
    ("f32", 50, "sell", 1024), ("f32", 64, "sell", 1536), ("f32", 79, "sell", 2048), ("f32", 80, *KERNELS)])
def test_scattered(contexts, precision, n, layout, rows):
    pr = W.linear(n)
    pr = W.renumbered(pr, np.random.default_rng(n).permutation(pr.mesh.nv), "scattered")
    _check(contexts, pr.mesh, pr.mu, pr.mask, pr.g, precision, (layout, rows))


def _split(pr, extra):
    """The problem with `extra` elements at each of a few nodes split at their
    centroid: rows of 14 + extra entries there."""
    t = np.asarray(pr.mesh.t, dtype=np.int64) - 1
    used = np.zeros(pr.mesh.nv, bool)
    pick = []
    for node in np.random.default_rng(extra).permutation(pr.mesh.nv):
        around = np.flatnonzero((t == node).any(axis=0))
        if around.size == 24 and not used[t[:, around]].any():
            used[t[:, around]] = True
            pick.extend(around[:extra])
        if len(pick) >= 3 * extra:
            break
    pick = np.array(pick)
    corner = t[:, pick]
    new = pr.mesh.nv + np.arange(pick.size)
    p = np.concatenate([pr.mesh.p, pr.mesh.p[:, corner].mean(axis=1)], axis=1)
    parts = [np.delete(t, pick, axis=1)]
    for k in range(4):
        c = corner.copy()
        c[k] = new
        parts.append(c)
    mu = np.concatenate([np.delete(pr.mu, pick)] + [pr.mu[pick]] * 4)
    t = np.concatenate(parts, axis=1)
    order = np.random.default_rng(1).permutation(p.shape[1])
    inv = np.argsort(order)
    p, t = np.asfortranarray(p[:, order]), np.asfortranarray((inv[t] + 1).astype(np.int32))
    fill = np.zeros(pick.size)
    mask = np.concatenate([pr.mask, fill.astype(np.uint8)])[order]
    return MESH(p=p, t=t, VE=element_volumes(p, t)), mu, mask, np.concatenate([pr.g, fill])[order]


# rows of up to 18 (20 with padding) and 26 entries
@pytest.mark.parametrize("precision,n,extra,layout,rows", [
    ("f64", 20, 4, "sell", 512), ("f64", 50, 4, "sell", 1024), ("f64", 64, 4, *KERNELS), ("f64", 20, 12, "sell", 512),
    ("f64", 50, 12, *KERNELS), ("f32", 20, 4, "sell", 512), ("f32", 50, 4, "sell", 1024), ("f32", 64, 4, "sell", 1536),
    ("f32", 79, 4, "sell", 2048), ("f32", 20, 12, "sell", 512), ("f32", 50, 12, "sell", 1024), ("f32", 64, 12, *KERNELS)])
def test_longer_rows(contexts, precision, n, extra, layout, rows):
    mesh, mu, mask, g = _split(W.linear(n), extra)
    _check(contexts, mesh, mu, mask, g, precision, (layout, rows))


@pytest.mark.parametrize("precision,dims,layout,rows", [
    ("f64", (30, 30, 600), "bricks", 2560), ("f64", (400, 400, 3), *KERNELS), ("f64", (230, 47, 55), "windows", 2560),
    ("f32", (400, 400, 3), "windows", 3072), ("f32", (230, 47, 55), "bricks", 5120)])
def test_grids(contexts, precision, dims, layout, rows):
    mesh = _box(*dims)
    rng = np.random.default_rng(5)
    mu = MU0 * rng.uniform(1.0, 50.0, mesh.nt)
    mask = ((mesh.p == 0.0) | (mesh.p == np.array(dims, float)[:, None])).any(axis=0)
    g = np.where(mask, rng.normal(size=mesh.nv), 0.0)
    _check(contexts, mesh, mu, mask.astype(np.uint8), g, precision, (layout, rows))


# rows of a Delaunay mesh of 700 nodes stay below 33 entries, of 9000 not
@pytest.mark.parametrize("points", [700, 9000])
def test_delaunay(contexts, points):
    from scipy.spatial import Delaunay

    rng = np.random.default_rng(points)
    pts = rng.random((points, 3))
    p = np.asfortranarray(pts.T)
    t = np.asfortranarray((Delaunay(pts).simplices.T + 1).astype(np.int32))
    t = np.asfortranarray(t[:, element_volumes(p, t) > 1e-9])
    mesh = MESH(p=p, t=t, VE=element_volumes(p, t))
    used = np.zeros(mesh.nv, bool)
    used[t.ravel() - 1] = True
    mask = ((~used) | (p[2] < 0.15) | (p[2] > 0.85)).astype(np.uint8)
    g = np.where(mask, p[2], 0.0)
    mu = MU0 * rng.uniform(1.0, 20.0, mesh.nt)
    for precision in ("f64", "f32"):
        _, _, launch, longest = _solve(contexts[0], mesh, mu, mask, g, precision)
        assert launch[0] == ("sell" if longest <= 32 else "kernels")


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("n,scattered", [(20, False), (63, False), (40, True)])
def test_three_kernels_in_graphs(contexts, n, scattered, precision):
    pr = W.linear(n)
    if scattered:
        pr = W.renumbered(pr, np.random.default_rng(n).permutation(pr.mesh.nv), "scattered")
    timed = Context(0)
    timed.set_timing(True)
    try:
        a, ra, la, _ = _solve(contexts[1], pr.mesh, pr.mu, pr.mask, pr.g, precision, 1e-10)
        b, rb, lb, _ = _solve(timed, pr.mesh, pr.mu, pr.mask, pr.g, precision, 1e-10)
        assert la == lb == ("kernels", 0, 0)
        assert np.array_equal(a, b) and ra == rb
        launches, ms = timed.spmv_timing()
        assert launches == rb.iterations and ms > 0.0
    finally:
        timed.close()


def test_trace(contexts, capfd, monkeypatch):
    """FEMEKO_HIP_TRACE=1 reports a refined solve on either path."""
    monkeypatch.setenv("FEMEKO_HIP_TRACE", "1")
    pr = W.linear(20)
    for ctx, text in zip(contexts, ("[fk trace] resident launch: iterations {} replacements {} ",
                                    "[fk trace] replacements {1} ")):
        _, rep, _, _ = _solve(ctx, pr.mesh, pr.mu, pr.mask, pr.g, "f32", 1e-10)
        assert text.format(rep.iterations, rep.outer) in capfd.readouterr().err


@pytest.mark.parametrize("boxes,nrhs,rows", [([(1, 1, 1)], 1, 512), ([(20, 20, 20)] * 3 + [(3, 4, 5)], 2, 512),
                                             ([(28, 28, 28)] * 7 + [(15, 15, 31), (2, 1, 3)], 3, 2048)])
def test_batch(contexts, boxes, nrhs, rows):
    rng = np.random.default_rng(nrhs)
    meshes = [_box(*b) for b in boxes]
    mus = [MU0 * rng.uniform(1.0, 5.0, m.nt) for m in meshes]
    masks = [np.zeros(m.nv, np.uint8) for m in meshes]
    for b, m in zip(boxes, masks):
        m[: (b[0] + 1) * 2] = 1
        m[-1] = 1
    gs = [np.where(m, rng.normal(size=(nrhs, m.size)), 0.0) for m in masks]
    out = []
    for ctx in contexts:
        b = Batch(meshes, nrhs=nrhs, ctx=ctx)
        try:
            b.set_coefficient(mus)
            b.assemble()
            b.set_dirichlet(masks, gs)
            assert b.solve_launch() == (0, 0)
            b.solve(rtol=1e-12)
            launch = b.solve_launch()
            assert launch[0] == rows and launch[1] >= 1 if ctx is contexts[0] else launch == (0, 0)
            out.append([b.potential(k) for k in range(b.nmesh)])
        finally:
            b.close()
    for u, v in zip(*out):
        assert np.linalg.norm(u - v) <= 1e-9 * np.linalg.norm(v)
