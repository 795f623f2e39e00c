"""Results copied to the caller's memory through the ring of pinned chunks
(transfer.hip): sizes at the edges of its ranges and chunks, aligned or not.
Copies are exact."""
import numpy as np
import pytest

from femeko_hip import workloads as W
from femeko_hip.device import Context, DeviceMesh
from test_gpu_resident import _box

pytestmark = pytest.mark.gpu


# nodes of 8 bytes: 512 KB and one plane less; 1 MB; 2 MB, a plane less and more
@pytest.mark.parametrize("cells", [(63, 31, 31), (63, 31, 30), (63, 63, 31), (63, 63, 63), (63, 63, 62), (63, 63, 64)])
def test_potential_round_trip(cells):
    mesh = _box(*cells)
    u = np.random.default_rng(mesh.nv).normal(size=mesh.nv)
    ctx = Context(0)
    dm = DeviceMesh(mesh, ctx)
    try:
        for _ in range(3):
            dm.set_potential(u)
            assert np.array_equal(dm.potential(), u)
    finally:
        dm.close()
        ctx.close()


@pytest.mark.parametrize("n", [31, 48, 63])
def test_field_large(n):
    """H in 4 to 36 MB and |H| in a third of it: |H| is the norm of each column of
    H (four roundings), whole and repeatable, also with two contexts."""
    pr = W.linear(n)
    ctxs = [Context(0), Context(0)]
    dms = [DeviceMesh(pr.mesh, c) for c in ctxs]
    try:
        u = np.random.default_rng(n).normal(size=pr.mesh.nv)
        out = []
        for dm in dms:
            dm.set_coefficient(pr.mu)
            dm.set_potential(u)
            H, Hn, _ = dm.field()
            assert np.allclose(np.sqrt((H * H).sum(axis=0)), Hn, rtol=1e-15 * 8, atol=0.0)
            assert np.array_equal(dm.get_coefficient(), pr.mu)
            out.append(H)
        assert np.array_equal(out[0], out[1])
    finally:
        for dm in dms:
            dm.close()
        for c in ctxs:
            c.close()
