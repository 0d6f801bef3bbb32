"""Point projections by waves and by sorted lanes give find_best's triangle and point, bit for bit."""
import numpy as np
import pytest

from parry_amd import TriMesh, scenes, split_projections

pytestmark = pytest.mark.gpu


def sphere(level):
    return scenes.noisy_icosphere(level, seed=3)


def plain_sphere(level):
    """No noise: many triangles at the same distance of the middle, ties at shared vertices and edges."""
    v, f = scenes.icosphere(level)
    return v.astype(np.float32), f.astype(np.uint32)


def grid(level):
    """A flat grid: boxes without thickness, whole-number coordinates."""
    n = 2 ** level
    x, y = np.meshgrid(np.arange(n + 1), np.arange(n + 1), indexing="ij")
    v = np.stack([x, y, np.zeros_like(x)], -1).reshape(-1, 3).astype(np.float32)
    i = (x[:-1, :-1] * (n + 1) + y[:-1, :-1]).reshape(-1)
    f = np.concatenate([np.stack([i, i + 1, i + n + 1], 1), np.stack([i + 1, i + n + 2, i + n + 1], 1)])
    return v, f.astype(np.uint32)


def slivers(level):
    """Stretched 1,000 times along x: no bound on the projections, so lanes only."""
    v, f = sphere(level)
    return v * np.array([1000.0, 1.0, 1.0], np.float32), f


def points_for(v, n, seed):
    rng = np.random.default_rng(seed)
    ext = np.abs(v).max()
    p = rng.uniform(-1.5, 1.5, (n, 3)).astype(np.float32) * ext
    k = n // 8
    p[:k] = v[rng.integers(0, len(v), k)]                                   # on vertices
    p[k:2 * k] = rng.normal(0.0, 1e-3, (k, 3)).astype(np.float32) * ext     # around the middle
    p[2 * k:3 * k] = np.round(p[2 * k:3 * k])
    special = np.array([[0, 0, 0], [np.nan, 0, 0], [np.inf, 0, 0], [0, -np.inf, 0], [1e30, 1e30, 1e30], [3e38, 0, 0],
                        [1e-42, 0, 0], [-0.0, 0, 0]], np.float32)
    m = min(len(special), n)
    p[n - m:] = special[:m]
    return p


@pytest.mark.parametrize("make,level,n", [(sphere, 0, 1), (sphere, 1, 64), (sphere, 4, 4097), (sphere, 5, 16384),
                                          (sphere, 5, 16385), (sphere, 3, 60001), (plain_sphere, 4, 5000),
                                          (plain_sphere, 4, 20000), (grid, 6, 3000), (grid, 6, 17000),
                                          (slivers, 4, 900), (slivers, 4, 17000)],
                         ids=lambda x: getattr(x, "__name__", str(x)))
def test_projection_mappings_match_oracle(orc, make, level, n):
    import torch

    v, f = make(level)
    p = points_for(v, n, level + n)
    print(f"case: {make.__name__} level {level}, {n} points", flush=True)
    mesh, ref_mesh = TriMesh(v, f), orc.OracleTriMesh(v, f)
    for solid in (False, True):
        out = mesh.project_local_points(torch.from_numpy(p).cuda(), solid)
        pt, inside, tri = (x.cpu().numpy() for x in split_projections(out))
        ref = ref_mesh.project_points(p, solid)
        assert np.array_equal(tri.view(np.uint32), ref["triangle"])
        hit = ref["triangle"] != 0xFFFFFFFF
        assert np.array_equal(pt[hit].view(np.uint32), ref["point"][hit].view(np.uint32))
        assert np.array_equal(inside[hit].astype(np.uint32), ref["is_inside"][hit])


def check_against_oracle(orc, v, f, p, solid=False):
    import torch

    out = TriMesh(v, f).project_local_points(torch.from_numpy(p).cuda(), solid)
    pt, inside, tri = (x.cpu().numpy() for x in split_projections(out))
    ref = orc.OracleTriMesh(v, f).project_points(p, solid)
    assert np.array_equal(tri.view(np.uint32), ref["triangle"])
    hit = ref["triangle"] != 0xFFFFFFFF
    assert np.array_equal(pt[hit].view(np.uint32), ref["point"][hit].view(np.uint32))
    assert np.array_equal(inside[hit].astype(np.uint32), ref["is_inside"][hit])


@pytest.mark.parametrize("n", [16384, 17000])
@pytest.mark.parametrize("scale", [1e-15, 1e-11, 1e-10, 3e-8, 1e-7, 1e8, 1e10, 1e15])
def test_projection_scales_match_oracle(orc, scale, n):
    """Edges from far below to just above the length that the projections' bound needs (products of
    four edges underflow), and meshes whose products overflow."""
    v, f = sphere(4)
    v = (v.astype(np.float64) * scale).astype(np.float32)
    p = (np.random.default_rng(n).uniform(-1.5, 1.5, (n, 3)) * scale).astype(np.float32)
    print(f"case: scale {scale}, {n} points", flush=True)
    check_against_oracle(orc, v, f, p)


@pytest.mark.parametrize("n", [64, 2561, 5121, 10241, 16384, 16385, 60001])
def test_far_and_nan_points_match_oracle(orc, n):
    """Points up to and beyond the distance that the bound on projections holds for, and points with a NaN: by a wave
    each, several to a wave and by sorted lanes."""
    v, f = sphere(4)
    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 3))
    p *= (10.0 ** rng.choice([0.0, 0.1, 0.5, 1.0, 1.7, 2.0, 2.3, 3.0, 5.0, 10.0, 17.0], n) /
          np.linalg.norm(p, axis=1))[:, None]
    p = p.astype(np.float32)
    p[rng.integers(0, n, n // 30), rng.integers(0, 3, n // 30)] = np.nan
    print(f"case: {n} points", flush=True)
    check_against_oracle(orc, v, f, p)


def test_more_long_walks_than_waves_take(orc):
    """140,000 points at the middle, all of whose walks are long: the plain walk's records (which the counted call
    gives), and the oracle's for some of them."""
    import torch

    v, f = sphere(5)
    p = np.random.default_rng(1).normal(0.0, 0.01, (140000, 3)).astype(np.float32)
    d = torch.from_numpy(p).cuda()
    mesh, counts = TriMesh(v, f), torch.zeros(140000, 2, dtype=torch.int32, device="cuda")
    print("case: 140,000 points", flush=True)
    got = mesh.project_local_points(d, False).view(torch.int32)
    want = mesh.project_local_points(d, False, counts=counts).view(torch.int32)
    assert int((counts[:, 0] > 256).sum()) > 131072
    assert torch.equal(got, want)
    ref = orc.OracleTriMesh(v, f).project_points(p[:2000], False)
    assert np.array_equal(got[:2000, 4].cpu().numpy().view(np.uint32), ref["triangle"])
