"""Workloads of the batched collision queries, one pass each through the public entry points.

A case names a kind of query and its sizes; ``prepare`` builds what a program holds before the call (meshes with
their Bvh, shape sets, poses, pair lists, output and work buffers), ``run`` makes the call.  The kinds are the
calls an engine built on this package makes: ray casts (single mesh, many meshes, with culling), point
projections, contacts over a broadphase's pairs, contact manifolds (fresh or carried over from the last frame),
shape casts, a mesh against shapes, the Bvh build, and a whole simulation frame.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from parry_amd import (
    Bvh,
    CONTACT_MANIFOLD_DTYPE,
    MeshContact,
    SHAPE_BALL,
    SHAPE_CAPSULE,
    SHAPE_CONE,
    SHAPE_CONVEX_POLYHEDRON,
    SHAPE_CUBOID,
    SHAPE_DESC_DTYPE,
    SHAPE_TRIANGLE,
    ShapeSet,
    TriMesh,
    TriMeshBatch,
    cast_shapes_pairs,
    cast_shapes_workspace_bytes,
    contact_manifolds_pfm,
    contact_manifolds_pfm_update,
    contact_manifolds_workspace_bytes,
    contact_pairs,
    contact_workspace_bytes,
    ploc_nodes,
    scenes,
    split_hits,
    split_projections,
)
from parry_amd.dynamics import DynamicScene

MAX_TOI = 10.0
# exact() tests every ray (or point) against every triangle: up to this many tests.
MOST_TESTS = 1 << 30

_MIXED = (SHAPE_CONVEX_POLYHEDRON, SHAPE_CUBOID, SHAPE_BALL, SHAPE_CAPSULE, SHAPE_CONE)
_TYPES = {
    "mixed": _MIXED,
    "polyhedra": (SHAPE_CONVEX_POLYHEDRON,),
    "cast": _MIXED + (SHAPE_TRIANGLE,),
    "features": (SHAPE_CUBOID, SHAPE_CAPSULE, SHAPE_CONE, SHAPE_TRIANGLE),
}


def listed():
    return [
        # A few sensor rays against one mesh, at the mesh's default mapping: latency and launches.
        {"name": "rays_1k", "kind": "rays", "rays": 1000, "level": 4, "mapping": "default", "culling": "none"},
        # A renderer's or lidar's batch against a mesh left as created.
        {"name": "rays_300k", "kind": "rays", "rays": 300007, "level": 5, "mapping": "default", "culling": "none"},
        # The benchmark's mesh and ray count at the mapping its autotuner picks there.
        {"name": "rays_1m", "kind": "rays", "rays": 1048576, "level": 6, "mapping": "binned", "culling": "none"},
        # Many objects of uneven sizes in one launch.
        {"name": "ray_batch", "kind": "ray_batch", "meshes": 12, "level": 6, "rays": 131072, "mapping": "binned"},
        # Distance queries of a cloth or particle step against a mesh.
        {"name": "points_260k", "kind": "points", "points": 262147, "level": 6, "solid": False},
        # One small island's pairs, every argument left at its default.
        {"name": "contact_300", "kind": "contact", "pairs": 300, "types": "mixed", "prediction": 0.01, "checked": True},
        # A granular frame of convex hulls.
        {"name": "contact_polyhedra", "kind": "contact", "pairs": 262144, "types": "polyhedra", "prediction": 0.01,
         "checked": False},
        # The largest pair list of the benchmark, five shape types.
        {"name": "contact_mixed_1m", "kind": "contact", "pairs": 1048576, "types": "mixed", "prediction": 0.01,
         "checked": False},
        # The solver's contact points for new pairs.
        {"name": "manifolds_250k", "kind": "manifolds", "pairs": 250001, "prediction": 0.02, "update": False},
        # Continuous collision detection of fast bodies.
        {"name": "casts_260k", "kind": "casts", "pairs": 262144, "target_distance": 0.0},
        # Bodies resting on terrain.
        {"name": "mesh_contact_32k", "kind": "mesh_contact", "shapes": 32768, "level": 6, "prediction": 0.01},
        # A whole frame: boxes, refit, pairs, contacts and motion of many bodies, replayed as a graph.
        {"name": "frame_260k", "kind": "frame", "shapes": 262144, "seeding": "plain"},
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rays", "rays", "ray_batch", "points", "contact", "contact", "manifolds", "manifolds", "casts",
                       "mesh_contact", "ploc", "frame"])
    if kind == "rays":
        return {"kind": kind, "rays": _log_size(rng, 60, 1000000), "level": rng.randint(2, 6),
                "mapping": rng.choice(["default", "default", "binned"]),
                "culling": rng.choice(["none", "none", "ignore_backfaces", "ignore_frontfaces"])}
    if kind == "ray_batch":
        return {"kind": kind, "meshes": rng.randint(2, 12), "level": rng.randint(3, 6),
                "rays": _log_size(rng, 2000, 130000), "mapping": rng.choice(["default", "binned"])}
    if kind == "points":
        return {"kind": kind, "points": _log_size(rng, 60, 260000), "level": rng.randint(2, 6),
                "solid": rng.random() < 0.5}
    if kind == "contact":
        return {"kind": kind, "pairs": _log_size(rng, 60, 1000000), "types": rng.choice(["mixed", "mixed", "polyhedra"]),
                "prediction": rng.choice([0.0, 0.01, 0.02, 0.1]), "checked": rng.random() < 0.5}
    if kind == "manifolds":
        return {"kind": kind, "pairs": _log_size(rng, 60, 250000), "prediction": rng.choice([0.0, 0.02, 0.1]),
                "update": rng.random() < 0.5}
    if kind == "casts":
        return {"kind": kind, "pairs": _log_size(rng, 60, 260000), "target_distance": rng.choice([0.0, 0.0, 0.05])}
    if kind == "mesh_contact":
        return {"kind": kind, "shapes": _log_size(rng, 60, 32000), "level": rng.randint(3, 6),
                "prediction": rng.choice([0.0, 0.01, 0.05])}
    if kind == "ploc":
        return {"kind": kind, "leaves": _log_size(rng, 60, 1000000)}
    return {"kind": kind, "shapes": _log_size(rng, 200, 260000), "seeding": rng.choice(["plain", "plain", "cache"])}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

_ICOSPHERES: dict = {}


def _mesh_arrays(level, seed, radius=1.0):
    """A noise-displaced icosphere (the subdivision, the same for every seed, is made once)."""
    if level not in _ICOSPHERES:
        _ICOSPHERES[level] = scenes.icosphere(level)
    v, f = _ICOSPHERES[level]
    r = np.random.default_rng(seed).uniform(-0.05, 0.05, v.shape[0])
    return (v * (radius * (1.0 + r))[:, None]).astype(np.float32), f.astype(np.uint32)


def _ray_inputs(case, seed):
    v, f = _mesh_arrays(case["level"], seed)
    return v, f, scenes.rays_into_unit_ball(case["rays"], seed + 1)


def _point_inputs(case, seed):
    v, f = _mesh_arrays(case["level"], seed)
    return v, f, np.random.default_rng(seed + 1).uniform(-1.5, 1.5, (case["points"], 3)).astype(np.float32)


def _batch_sizes(case):
    """Levels over [2, level] (one of them the largest) and uneven ray counts, the mean about the case's."""
    rng = np.random.default_rng([case["meshes"], case["level"], case["rays"]])
    levels = rng.integers(2, case["level"] + 1, case["meshes"])
    levels[0] = case["level"]
    counts = np.maximum(1, np.rint(case["rays"] * np.exp2(rng.uniform(-3.0, 1.0, case["meshes"])))).astype(np.int64)
    return levels, counts


def _shapes(n, types, seed, scale=1.0):
    """``n`` shapes, types uniform: hulls of 8 to 64 points (a pool of 128, each stretched per axis), and the other
    types with the sizes of ``scenes.mixed_shapes``."""
    rng = np.random.default_rng(seed)
    pool = [scenes.convex_hull_vertices(scenes.convex_point_cloud(rng, int(rng.integers(8, 65)))) for _ in range(128)]
    pool_first = np.cumsum([0] + [p.shape[0] for p in pool])
    pool_v = np.concatenate(pool, 0)
    t = np.asarray(types)[rng.integers(0, len(types), n)]
    d = np.zeros(n, SHAPE_DESC_DTYPE)
    d["type"] = t
    sizes = rng.uniform(0.5, 1.5, (n, 3)) * scale
    d["params"][t == SHAPE_CUBOID, :3] = sizes[t == SHAPE_CUBOID]
    d["params"][t == SHAPE_BALL, 0] = sizes[t == SHAPE_BALL, 0]
    d["params"][t == SHAPE_CAPSULE, :2] = sizes[t == SHAPE_CAPSULE, :2] * [1.0, 0.5]
    d["params"][t == SHAPE_CONE, :2] = sizes[t == SHAPE_CONE, :2]
    counts = np.zeros(n, np.int64)
    hull = np.nonzero(t == SHAPE_CONVEX_POLYHEDRON)[0]
    which = rng.integers(0, len(pool), hull.size)
    counts[hull] = np.diff(pool_first)[which]
    counts[t == SHAPE_TRIANGLE] = 3
    first = np.cumsum(counts) - counts
    verts = (rng.normal(0.0, 0.7, (int(counts.sum()), 3)) * scale).astype(np.float32)
    if hull.size:
        at = np.arange(int(counts[hull].sum())) - np.repeat(np.cumsum(counts[hull]) - counts[hull], counts[hull])
        stretch = np.repeat(rng.uniform(0.9, 1.1, (hull.size, 3)) * scale, counts[hull], axis=0)
        verts[np.repeat(first[hull], counts[hull]) + at] = pool_v[np.repeat(pool_first[which], counts[hull]) + at] * stretch
    d["num_vertices"] = counts
    d["first_vertex"] = np.where(counts > 0, first, 0)
    return d, verts


def _cuda(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def _scene(n, types, seed):
    """Shapes at random rotations in a cube where each box overlaps eight others on average."""
    rng = np.random.default_rng(seed + 1)
    descs, verts = _shapes(n, types, seed)
    poses = np.concatenate([scenes.random_rotations(n, rng), np.zeros((n, 3))], 1).astype(np.float32)
    shapes = ShapeSet(descs, verts)
    boxes = shapes.compute_aabbs(_cuda(poses)).cpu().numpy()
    side = scenes.calibrate_cube_side((boxes[:, 3:] - boxes[:, :3]) * 0.5, min(8.0, 0.25 * n), rng, samples=20000)
    poses[:, 4:] = rng.uniform(0.0, side, (n, 3))
    return shapes, descs, verts, poses


def _near_pairs(n, types, seed, spread, scale=1.0):
    """Shapes 2q and 2q + 1, the second at N(0, spread) per axis from the first."""
    rng = np.random.default_rng(seed + 1)
    descs, verts = _shapes(2 * n, types, seed, scale)
    poses = np.concatenate([scenes.random_rotations(2 * n, rng), np.zeros((2 * n, 3))], 1)
    poses[0::2, 4:] = rng.uniform(-40.0, 40.0, (n, 3))
    poses[1::2, 4:] = poses[0::2, 4:] + rng.normal(0.0, spread, (n, 3))
    pairs = torch.arange(2 * n, dtype=torch.int32, device="cuda").reshape(n, 2)
    return descs, verts, poses, pairs, rng


def _set_mapping(mesh, mapping):
    if mapping == "binned":
        mesh.set_tuning("binned", block_size=128)


def _empty(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "rays":
        v, f, rays = _ray_inputs(case, seed)
        s["mesh"], s["rays"], s["out"] = TriMesh(v, f), _cuda(rays), _empty(case["rays"], 5)
        _set_mapping(s["mesh"], case["mapping"])
    elif kind == "ray_batch":
        levels, counts = _batch_sizes(case)
        s["batch"] = TriMeshBatch([TriMesh(*_mesh_arrays(int(l), seed + k)) for k, l in enumerate(levels)], counts)
        s["rays"] = _cuda(scenes.rays_into_unit_ball(int(counts.sum()), seed + 1))
        s["out"] = _empty(int(counts.sum()), 5)
        _set_mapping(s["batch"], case["mapping"])
    elif kind == "points":
        v, f, points = _point_inputs(case, seed)
        s["mesh"], s["points"], s["out"] = TriMesh(v, f), _cuda(points), _empty(case["points"], 5)
    elif kind == "contact":
        s["shapes"], _, _, poses = _scene(case["pairs"] // 3 + 16, _TYPES[case["types"]], seed)
        s["poses"] = _cuda(poses)
        boxes = s["shapes"].compute_aabbs(s["poses"])
        s["pairs"] = Bvh.from_leaves(boxes, "ploc").self_pairs()[: case["pairs"]].contiguous()
        m = s["pairs"].shape[0]
        s["out"], s["workspace"] = None, None
        if not case["checked"]:  # a program that trusts its pairs keeps its buffers too
            s["out"] = _empty(m, 14)
            s["workspace"] = torch.empty(contact_workspace_bytes(m), dtype=torch.uint8, device="cuda")
    elif kind == "manifolds":
        n = case["pairs"]
        descs, verts, poses, s["pairs"], rng = _near_pairs(n, _TYPES["features"], seed, 0.6, 0.7)
        s["shapes"], s["poses"] = ShapeSet(descs, verts), _cuda(poses)
        s["out"] = _empty(n, CONTACT_MANIFOLD_DTYPE.itemsize, dtype=torch.uint8)
        s["workspace"] = torch.empty(contact_manifolds_workspace_bytes(n), dtype=torch.uint8, device="cuda")
        if case["update"]:  # bodies that sway between two frames
            poses[:, 4:] += rng.normal(0.0, 1.0e-4, (2 * n, 3))
            s["sway"] = [s["poses"], _cuda(poses)]
            s["frame"] = 0
            contact_manifolds_pfm(s["shapes"], s["poses"], s["pairs"], case["prediction"], out=s["out"],
                                  workspace=s["workspace"], check_indices=False)
    elif kind == "casts":
        n = case["pairs"]
        descs, verts, poses, s["pairs"], rng = _near_pairs(n, _TYPES["cast"], seed, 0.0)
        d = rng.normal(0.0, 1.0, (n, 3))
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        poses[1::2, 4:] += d * rng.uniform(2.0, 6.0, (n, 1))
        vels = rng.uniform(-0.3, 0.3, (2 * n, 3))
        vels[1::2] += (-d + rng.normal(0.0, 0.3, (n, 3))) * rng.uniform(0.5, 3.0, (n, 1))
        s["shapes"], s["poses"], s["vels"] = ShapeSet(descs, verts), _cuda(poses), _cuda(vels)
        s["out"] = _empty(n, 14)
        s["workspace"] = torch.empty(cast_shapes_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    elif kind == "mesh_contact":
        n = case["shapes"]
        rng = np.random.default_rng(seed + 1)
        descs, verts = _shapes(n, _MIXED, seed, 0.15)
        d = rng.normal(0.0, 1.0, (n, 3))
        d *= 8.0 * rng.uniform(0.96, 1.04, (n, 1)) / np.linalg.norm(d, axis=1, keepdims=True)
        s["contact"] = MeshContact(TriMesh(*_mesh_arrays(case["level"], seed, 8.0)), ShapeSet(descs, verts))
        s["mesh_pose"] = _cuda([0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0])
        s["poses"] = _cuda(np.concatenate([scenes.random_rotations(n, rng), d], 1))
        s["capacity"] = 64 * n + 1024
        s["out"], s["triangles"] = _empty(n, 14), _empty(n, dtype=torch.int32)
        s["workspace"] = torch.empty(s["contact"].workspace_bytes(s["capacity"]), dtype=torch.uint8, device="cuda")
        s["needed"] = _empty(1, dtype=torch.int64)
    elif kind == "ploc":
        rng = np.random.default_rng(seed)
        n = case["leaves"]
        c = rng.uniform(0.0, 2.0 * n ** (1.0 / 3.0), (n, 3))
        h = rng.uniform(0.3, 1.5, (n, 3))
        s["aabbs"], s["out"] = _cuda(np.concatenate([c - h, c + h], 1)), _empty(max(1, n - 1), 64, dtype=torch.uint8)
    else:
        n = case["shapes"]
        shapes, descs, verts, poses = _scene(n, _MIXED, seed)
        scene = DynamicScene(descs, verts, poses, seed=seed, seeding=case["seeding"])
        scene.contacts.zero_()
        scene.capture()
        s["scene"], s["start"] = scene, scene.poses.clone()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _records(out):
    """The values and the status word of (m, 14) contact or cast records (views)."""
    return out[:, :13], out.view(torch.int32)[:, 13]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "rays":
        if case["culling"] == "none":
            return split_hits(s["mesh"].cast_local_rays_and_get_normal(s["rays"], MAX_TOI, True, out=s["out"]))
        return split_hits(s["mesh"].cast_local_rays_with_culling(s["rays"], MAX_TOI, case["culling"], out=s["out"]))
    if kind == "ray_batch":
        return split_hits(s["batch"].cast_local_rays_and_get_normal(s["rays"], MAX_TOI, True, out=s["out"]))
    if kind == "points":
        return split_projections(s["mesh"].project_local_points(s["points"], case["solid"], out=s["out"]))
    if kind == "contact":
        return _records(contact_pairs(s["shapes"], s["poses"], s["pairs"], case["prediction"], out=s["out"],
                                      workspace=s["workspace"], check_indices=case["checked"]))
    if kind == "manifolds":
        if case["update"]:
            s["frame"] ^= 1
            return contact_manifolds_pfm_update(s["shapes"], s["sway"][s["frame"]], s["pairs"], case["prediction"],
                                                s["out"], workspace=s["workspace"], check_indices=False)
        return contact_manifolds_pfm(s["shapes"], s["poses"], s["pairs"], case["prediction"], out=s["out"],
                                     workspace=s["workspace"], check_indices=False)
    if kind == "casts":
        return _records(cast_shapes_pairs(s["shapes"], s["poses"], s["vels"], s["pairs"],
                                          target_distance=case["target_distance"], out=s["out"],
                                          workspace=s["workspace"], check_indices=False))
    if kind == "mesh_contact":
        out, triangles, needed = s["contact"].contact(s["mesh_pose"], s["poses"], case["prediction"], s["capacity"],
                                                      out=s["out"], triangles=s["triangles"],
                                                      workspace=s["workspace"], needed=s["needed"])
        return _records(out) + (triangles, needed)
    if kind == "ploc":
        return ploc_nodes(s["aabbs"], out=s["out"])
    # A frame from the state the program holds: the poses it sets, then the captured step.
    scene = s["scene"]
    with torch.cuda.stream(scene.stream):
        scene.poses.copy_(s["start"])
    scene.step()
    torch.cuda.current_stream().wait_stream(scene.stream)
    return (scene.poses, scene.pairs, scene.count) + _records(scene.contacts)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

# Bytes of one shape: its pose (28), its record (32) and, for one in five of the mixed types, 27 vertices of 12.
_SHAPE_BYTES = {"mixed": 125, "polyhedra": 384, "cast": 120, "features": 69}


def _mesh_bytes(level, queries):
    """The mesh's nodes and triangles once, or less where so few queries cannot touch them all (a path to a leaf
    per query)."""
    tris = 20 * 4 ** level
    return min(112 * tris, queries * (64 * int(math.log2(tris)) + 48))


def work(case):
    kind = case["kind"]
    if kind == "rays":
        return {"bytes": 44 * case["rays"] + _mesh_bytes(case["level"], case["rays"]), "flops": 0}
    if kind == "ray_batch":
        levels, counts = _batch_sizes(case)
        meshes = sum(_mesh_bytes(int(l), int(c)) for l, c in zip(levels, counts))
        return {"bytes": 44 * int(counts.sum()) + meshes, "flops": 0}
    if kind == "points":
        return {"bytes": 32 * case["points"] + _mesh_bytes(case["level"], case["points"]), "flops": 0}
    if kind == "contact":
        return {"bytes": case["pairs"] * (8 + 56 + _SHAPE_BYTES[case["types"]] / 3), "flops": 0}
    if kind == "manifolds":
        # header, 8 bytes of pair and about 2.7 points of 36 bytes for two pairs in three
        points = 32 + 8 + 65 + (97 if case["update"] else 0)
        return {"bytes": case["pairs"] * (points + 2 * _SHAPE_BYTES["features"]), "flops": 0}
    if kind == "casts":
        return {"bytes": case["pairs"] * (8 + 56 + 24 + 2 * _SHAPE_BYTES["cast"]), "flops": 0}
    if kind == "mesh_contact":
        return {"bytes": case["shapes"] * (_SHAPE_BYTES["mixed"] + 60) + _mesh_bytes(case["level"], 27 * case["shapes"]),
                "flops": 0}
    if kind == "ploc":
        return {"bytes": case["leaves"] * (24 + 64), "flops": 0}
    # boxes, a refit tree, three and a half pairs with their contacts, and the poses' motion per shape
    return {"bytes": case["shapes"] * (_SHAPE_BYTES["mixed"] + 24 + 64 + 3.5 * (8 + 56) + 28 + 24), "flops": 0}


def tolerance(case):
    """Every query evaluates parry's sequence of 32-bit operations without contraction, and its tests hold it to the
    same bits: indices, statuses and trees follow from comparisons of those values, so another order of the same
    operations would not be correct."""
    return "exact"


# ---------------------------------------------------------------------------
# 64-bit answers by testing every triangle
# ---------------------------------------------------------------------------

def _triangles64(v, f):
    t = torch.from_numpy(v.astype(np.float64)[f.astype(np.int64)]).cuda()
    return t[:, 0], t[:, 1], t[:, 2]


def _dot(a, b):
    return (a * b).sum(-1)


def _exact_rays(case, seed):
    v, f, rays = _ray_inputs(case, seed)
    a, b, c = _triangles64(v, f)
    n = torch.linalg.cross(b - a, c - a)
    r = torch.from_numpy(rays.astype(np.float64)).cuda()
    toi, normal = torch.zeros(len(r), dtype=torch.float64), torch.zeros(len(r), 3, dtype=torch.float64)
    step = max(1, (1 << 23) // len(a))
    for i in range(0, len(r), step):
        o, d = r[i:i + step, None, :3], r[i:i + step, None, 3:]
        dn = _dot(d, n)
        t = _dot(a - o, n) / dn
        p = o + d * t[..., None]
        inside = (t >= 0) & (t <= MAX_TOI)
        for x, y in ((a, b), (b, c), (c, a)):
            inside &= _dot(torch.linalg.cross((y - x).expand_as(p), p - x), n.expand_as(p)) >= -1e-13
        if case["culling"] != "none":
            inside &= (dn < 0) if case["culling"] == "ignore_backfaces" else (dn > 0)
        best, at = torch.where(inside, t, torch.inf).min(1)
        hit = torch.isfinite(best)
        m = torch.nn.functional.normalize(n[at], dim=1)
        m = m * -torch.sign(_dot(m, r[i:i + step, 3:]))[:, None]
        toi[i:i + step] = torch.where(hit, best, 0.0).cpu()
        normal[i:i + step] = torch.where(hit[:, None], m, 0.0).cpu()
    return toi, normal, None


def _exact_points(case, seed):
    v, f, points = _point_inputs(case, seed)
    a, b, c = _triangles64(v, f)
    n = torch.linalg.cross(b - a, c - a)
    pts = torch.from_numpy(points.astype(np.float64)).cuda()
    out = torch.zeros(len(pts), 3, dtype=torch.float64)
    step = max(1, (1 << 22) // len(a))
    for i in range(0, len(pts), step):
        p = pts[i:i + step, None, :]
        q = p - n * (_dot(p - a, n) / _dot(n, n))[..., None]
        inside = torch.ones(q.shape[:2], dtype=torch.bool, device=q.device)
        best, where = torch.full(q.shape[:2], torch.inf, dtype=torch.float64, device=q.device), q.clone()
        for x, y in ((a, b), (b, c), (c, a)):
            e = y - x
            inside &= _dot(torch.linalg.cross(e.expand_as(q), q - x), n.expand_as(q)) >= 0
            on = x + e * (_dot(p - x, e) / _dot(e, e)).clamp(0.0, 1.0)[..., None]
            dist = _dot(p - on, p - on)
            where = torch.where((dist < best)[..., None], on, where)
            best = torch.minimum(best, dist)
        where = torch.where(inside[..., None], q, where)
        best = torch.where(inside, _dot(p - q, p - q), best)
        at = best.argmin(1)
        out[i:i + step] = where[torch.arange(len(at), device=at.device), at].cpu()
    return out, None, None


def exact(case, seed):
    """Rays and points by every triangle in 64 bits.  The other queries' results are where parry's 32-bit iteration
    stops (or whole numbers): the same iteration in 64 bits stops elsewhere, so they have no such value."""
    if case["kind"] == "rays" and case["rays"] * 20 * 4 ** case["level"] <= MOST_TESTS:
        return _exact_rays(case, seed)
    if case["kind"] == "points" and not case["solid"] and case["points"] * 20 * 4 ** case["level"] <= MOST_TESTS:
        return _exact_points(case, seed)
    return None
