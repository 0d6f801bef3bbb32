"""The mesh contact's counting pass keeps a shape's first triangles and its writing
pass walks again for shapes with more: capacities at which the number kept is
none, below, between and above what the shapes have, and shapes with more than
it ever keeps (256).  The contacts and the candidate count are the oracle's
(contact_composite_shape_shape.rs:14-59), unchanged where the capacity suffices."""
import numpy as np
import pytest

from parry_amd import (
    PQ_CONTACT_TRUNCATED,
    SHAPE_BALL,
    SHAPE_CUBOID,
    SHAPE_DESC_DTYPE,
    MeshContact,
    ShapeSet,
    TriMesh,
    scenes,
)

pytestmark = pytest.mark.gpu
IDENT = np.array([0, 0, 0, 1, 0, 0, 0], np.float32)


def _shapes():
    """A ball over most of the mesh, a cuboid over part of it, small ones and one apart."""
    d = np.zeros(6, SHAPE_DESC_DTYPE)
    d["type"] = [SHAPE_BALL, SHAPE_CUBOID, SHAPE_BALL, SHAPE_CUBOID, SHAPE_BALL, SHAPE_BALL]
    for i, p in enumerate([(1.5,), (0.5, 0.4, 0.3), (0.3,), (0.05, 0.1, 0.1), (0.02,), (0.1,)]):
        d["params"][i][:len(p)] = p
    poses = np.tile(IDENT, (6, 1))
    poses[:, 4:] = [(0.5, 0, 0), (2, 0, 0), (0, 2, 0), (0, 0, 2), (0, -2, 0), (9, 9, 9)]
    return d, poses


@pytest.mark.parametrize("extra", [0, 1, 700])
def test_kept_and_walked_again(orc, extra):
    import torch

    v, f = scenes.noisy_icosphere(4, seed=2, radius=2.0)
    mesh, om = TriMesh(v, f), orc.OracleTriMesh(v, f)
    descs, poses = _shapes()
    descs, poses = np.concatenate([descs, descs[5:].repeat(extra)]), np.concatenate([poses, poses[5:].repeat(extra, 0)])
    verts = np.zeros((0, 3), np.float32)
    mc = MeshContact(mesh, ShapeSet(descs, verts))
    ref = om.contact_shapes(IDENT, descs, verts, poses, 0.02)
    counts = np.array([om.contact_shapes(IDENT, descs[q:q + 1], verts, poses[q:q + 1], 0.02)["candidates"]
                       for q in range(6)] + [0] * extra, np.int64)
    assert counts.max() > 256 and counts[1] > counts[2] > counts[4] >= 1, counts[:6]
    ends, total = np.cumsum(counts), int(counts.sum())
    n, mp, p = len(descs), torch.from_numpy(IDENT).cuda(), torch.from_numpy(poses).cuda()
    # 14 * capacity / n triangles are kept per shape, at most 256
    caps = {0, 1, n // 14, n // 14 + 1, (int(counts[4]) * n + 13) // 14, (int(counts[2]) * n + 13) // 14,
            (int(counts[2]) * n - 1) // 14, (256 * n) // 14 + 1, total - 1, total, 2 * total}
    for cap in sorted(caps):
        print(f"case: kept candidates, {n} shapes, capacity {cap} of {total}", flush=True)
        out, tri, needed = mc.contact(mp, p, 0.02, cap)
        torch.cuda.synchronize()
        o, tri = out.cpu().numpy(), tri.cpu().numpy().view(np.uint32)
        has = o.view(np.uint32)[:, 13]
        assert int(needed.item()) == total == ref["candidates"]
        short = (ends > cap) & (counts > 0)
        assert (has[short] == PQ_CONTACT_TRUNCATED).all()
        assert np.array_equal(has[~short], ref["status"][~short].astype(np.uint32))
        c = ~short & (ref["status"] == 1)
        assert np.array_equal(tri[c], ref["triangle"][c])
        err = np.abs(o[c, :13] - ref["out"][c]) / np.maximum(1.0, np.abs(ref["out"][c]))
        assert err.max(initial=0) <= 1e-5  # the bar of the other mesh contact tests
