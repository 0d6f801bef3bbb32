"""EPA's face choice without a heap, and its polytopes' way through the tiers, against the oracle.

The tiers take the next face as the maximum of the face keys and only rebuild parry's heap when several live
faces share it: symmetric shapes at aligned poses share it all the time.  Long runs (curved shapes, deep
overlaps) cross the tiers' vertex and face limits."""
import numpy as np
import pytest

from parry_amd import SHAPE_DESC_DTYPE, ShapeSet, contact_pairs

pytestmark = pytest.mark.gpu

# quaternions of quarter turns (i, j, k, w)
TURNS = np.array([[0, 0, 0, 1], [1, 0, 0, 0], [0, 1, 0, 0], [0.5, 0.5, 0.5, 0.5], [0, 0.70710678, 0, 0.70710678],
                  [0.70710678, 0, 0, 0.70710678]], np.float64)
OCTAHEDRON = np.array([[1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1]], np.float32)


def aligned_case(types, n, seed):
    """``n`` pairs of unit shapes of the two types at quarter turns, offset by multiples of a quarter."""
    rng = np.random.default_rng(seed)
    d = np.zeros(2 * n, SHAPE_DESC_DTYPE)
    d["type"] = np.tile(types, n)
    d["params"][:, :3] = 1.0
    d["params"][d["type"] == 2, 1] = 0.5
    poly = d["type"] == 4
    d["num_vertices"][poly] = len(OCTAHEDRON)
    d["params"][poly] = 0.0
    poses = np.zeros((2 * n, 7))
    poses[:, :4] = TURNS[rng.integers(0, len(TURNS), 2 * n)]
    poses[1::2, 4:] = rng.integers(-5, 6, (n, 3)) * 0.25
    return d, OCTAHEDRON, poses.astype(np.float32), np.arange(2 * n, dtype=np.uint32).reshape(n, 2)


def deep_case(types, n, seed):
    """``n`` pairs of curved shapes with centres close together: up to parry's 100 iterations."""
    rng = np.random.default_rng(seed)
    d = np.zeros(2 * n, SHAPE_DESC_DTYPE)
    d["type"] = np.tile(types, n)
    d["params"][:, :2] = rng.uniform(0.3, 1.5, (2 * n, 2))
    d["params"][:, 2] = 1.0
    q = rng.standard_normal((2 * n, 4))
    poses = np.concatenate([q / np.linalg.norm(q, axis=1, keepdims=True), np.zeros((2 * n, 3))], 1)
    poses[1::2, 4:] = rng.normal(0.0, 0.2, (n, 3))
    return d, np.zeros((0, 3), np.float32), poses.astype(np.float32), np.arange(2 * n, dtype=np.uint32).reshape(n, 2)


CASES = [(aligned_case, t) for t in ((1, 1), (1, 4), (4, 4), (1, 2), (2, 2), (3, 3), (1, 3))]
CASES += [(deep_case, t) for t in ((2, 2), (2, 3), (3, 3), (1, 2))]


@pytest.mark.parametrize("make,types", CASES, ids=lambda v: getattr(v, "__name__", str(v)))
def test_epa_tiers_match_oracle(orc, make, types):
    import torch

    for n in (1, 7, 1500):
        descs, verts, poses, pairs = make(types, n, 7 + n)
        print(f"case: {make.__name__} {types}, {n} pairs", flush=True)
        shapes = ShapeSet(descs, verts)
        out, iters = contact_pairs(shapes, torch.from_numpy(poses).cuda(),
                                   torch.from_numpy(pairs.view(np.int32)).cuda(), 0.25, with_iters=True)
        out, iters = out.cpu().numpy(), iters.cpu().numpy()
        ref = orc.contact_pairs(descs, verts, poses, pairs, 0.25)
        has = out.view(np.uint32)[:, 13].astype(np.int64)
        assert np.array_equal(has, ref["status"])
        hit = has == 1
        # parry's own sequence of f32 operations: the same bits (+0.0: signed zeros compare equal)
        assert np.array_equal(out[hit, :13] + 0.0, ref["out"][hit] + 0.0)
        assert np.array_equal(iters[:, 0], ref["iters"][:, 0].astype(np.int32))
        print(f"  {hit.sum()} contacts, EPA iterations up to {ref['iters'][:, 1].max()}")


@pytest.mark.parametrize("m", [16384, 16385])
@pytest.mark.parametrize("make,types", CASES, ids=lambda v: getattr(v, "__name__", str(v)))
def test_many_pairs_match_few(make, types, m):
    """Up to 16,384 pairs take more lanes per pair in the first two tiers: the same records on both sides."""
    import torch

    print(f"case: {make.__name__} {types}, {m} pairs", flush=True)
    n = 700
    descs, verts, poses, pairs = make(types, n, 3)
    shapes, poses = ShapeSet(descs, verts), torch.from_numpy(poses).cuda()
    few = torch.from_numpy(pairs.view(np.int32)).cuda()
    want, wi = contact_pairs(shapes, poses, few, 0.25, with_iters=True)
    pick = torch.from_numpy(np.random.default_rng(4).integers(0, n, m)).cuda()
    out, it = contact_pairs(shapes, poses, few[pick].contiguous(), 0.25, with_iters=True)
    assert torch.equal(out.view(torch.int32), want[pick].view(torch.int32))
    assert torch.equal(it, wi[pick])


@pytest.mark.parametrize("m,count", [(131071, None), (131072, None), (131072, 1), (140001, 131000), (135169, 0)])
def test_ordered_pairs_match_unordered(m, count):
    """From 131,072 pairs of several shape types on, the pairs are taken class by class: every pair's record is the
    one a small call writes, and slots at or beyond a device-side count are left alone."""
    import ctypes

    import torch

    from parry_amd import _native, contact_workspace_bytes, scenes

    print(f"case: {m} mixed pairs, count {count}", flush=True)
    sc = scenes.mixed_scene(900, seed=5)
    n = 4000
    rng = np.random.default_rng(2)
    base = rng.integers(0, 900, (n, 2)).astype(np.int32)
    shapes, poses = ShapeSet(sc["descs"], sc["vertices"]), torch.from_numpy(sc["poses"]).cuda()
    want = contact_pairs(shapes, poses, torch.from_numpy(base).cuda(), 0.5, check_indices=False)
    pick = torch.from_numpy(rng.integers(0, n, m)).cuda()
    pairs = torch.from_numpy(base).cuda()[pick].contiguous()
    out = torch.full((m, 14), -7.0, device="cuda")
    if count is None:
        contact_pairs(shapes, poses, pairs, 0.5, out=out, check_indices=False)
    else:
        ws = torch.empty(contact_workspace_bytes(m), dtype=torch.uint8, device="cuda")
        dev_count = torch.tensor([count], dtype=torch.int64, device="cuda")
        _native.check(_native.lib().pq_contact_pairs_device_count(
            shapes.handle, poses.data_ptr(), pairs.data_ptr(), m, dev_count.data_ptr(), 0.5, None, out.data_ptr(), None,
            ws.data_ptr(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    k = m if count is None else count
    assert torch.equal(out[:k].view(torch.int32), want[pick[:k]].view(torch.int32))
    assert bool((out[k:] == -7.0).all())


@pytest.mark.parametrize("k", [0, 1, 2, 5, 9, 33])
def test_few_overlaps_match_oracle(orc, k):
    """Lists shorter than a tier's waves, down to empty ones: k overlapping pairs of 40, and of 16,400."""
    import torch

    print(f"case: {k} overlapping pairs", flush=True)
    descs, verts, poses, pairs = deep_case((2, 3), 40, 11)
    poses[2 * k + 1::2, 4] += 50.0
    ref = orc.contact_pairs(descs, verts, poses, pairs, 0.25)
    shapes, d = ShapeSet(descs, verts), torch.from_numpy(poses).cuda()
    few = torch.from_numpy(pairs.view(np.int32)).cuda()
    out, iters = contact_pairs(shapes, d, few, 0.25, with_iters=True)
    hit = ref["status"] == 1
    assert hit.sum() == k and np.array_equal(out.cpu().numpy().view(np.uint32)[:, 13], ref["status"])
    assert np.array_equal(out.cpu().numpy()[hit, :13] + 0.0, ref["out"][hit] + 0.0)
    pick = torch.full((16400,), 39, device="cuda")
    pick[torch.arange(40, device="cuda") * 400] = torch.arange(40, device="cuda")
    many, it = contact_pairs(shapes, d, few[pick].contiguous(), 0.25, with_iters=True)
    assert torch.equal(many.view(torch.int32), out.view(torch.int32)[pick])
    assert torch.equal(it, iters[pick])
