"""The buffers of large point projections (TriMesh::project_local_point,
point_composite_shape.rs:164-168): their own, safe under captured graphs, growth,
several threads and more points than one sort takes."""
import ctypes
import threading

import numpy as np
import pytest

from parry_amd import Graph, TriMesh, _native, scenes

pytestmark = pytest.mark.gpu


def cloud(n, seed):
    import torch

    return torch.from_numpy(np.random.default_rng(seed).uniform(-1.5, 1.5, (n, 3)).astype(np.float32)).cuda()


def captured(stream, issue, keep):
    """What ``issue`` launches on ``stream``, as a graph."""
    handle, sp = ctypes.c_void_p(), ctypes.c_void_p(stream.cuda_stream)
    _native.check(_native.lib().pq_stream_begin_capture(sp))
    try:
        issue()
    finally:
        _native.check(_native.lib().pq_stream_end_capture(sp, ctypes.byref(handle)))
    return Graph(handle, keep=keep)


def test_ray_graph_survives_larger_projections():
    """A graph of binned rays replays the same hits after and between projections of more points on its stream,
    whose buffers grow, and with projections on its stream beside replays on another."""
    import torch

    mesh = TriMesh(*scenes.noisy_icosphere(5, 1))
    mesh.set_tuning("binned", block_size=128)
    rays = torch.from_numpy(scenes.rays_into_unit_ball(30000, 2)).cuda()
    s, other = torch.cuda.Stream(), torch.cuda.Stream()
    want = mesh.cast_local_rays_and_get_normal(rays, 10.0, True).view(torch.int32).clone()
    out = torch.zeros(30000, 5, device="cuda")
    torch.cuda.synchronize()
    mesh.cast_local_rays_and_get_normal(rays, 10.0, True, out=out, stream=s)  # the buffers, before the capture
    graph = captured(s, lambda: mesh.cast_local_rays_and_get_normal(rays, 10.0, True, out=out, stream=s), (mesh, out))
    for n in (17000, 40000, 300000, 20000):
        p, first = cloud(n, n), None
        torch.cuda.synchronize()
        for replay in range(3):
            print(f"case: {n} points, replay {replay}", flush=True)
            out.zero_()
            torch.cuda.synchronize()
            got = mesh.project_local_points(p, True, stream=s)
            graph.launch(s if replay < 2 else other)
            again = mesh.project_local_points(p, True, stream=s)
            torch.cuda.synchronize()
            assert torch.equal(out.view(torch.int32), want)
            first = got.view(torch.int32) if first is None else first
            assert torch.equal(got.view(torch.int32), first) and torch.equal(again.view(torch.int32), first)


def test_captured_projection_and_capture_beside_growth():
    """A large projection inside a capture gives the eager call's records on every replay; a first large projection on
    another stream does not end the capture."""
    import torch

    mesh = TriMesh(*scenes.noisy_icosphere(4, 1))
    p, q = cloud(20000, 1), cloud(50000, 2)
    want = mesh.project_local_points(p, False).view(torch.int32).clone()
    beside = mesh.project_local_points(q, False).view(torch.int32).clone()
    out, out2 = torch.zeros(20000, 5, device="cuda"), torch.zeros(50000, 5, device="cuda")
    s, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()

    def issue():
        mesh.project_local_points(p, False, out=out, stream=s)
        mesh.project_local_points(q, False, out=out2, stream=other)

    print("case: capture of 20,000 points with 50,000 beside it", flush=True)
    graph = captured(s, issue, (mesh, p, out))
    torch.cuda.synchronize()
    assert torch.equal(out2.view(torch.int32), beside)
    for replay in range(3):
        print(f"case: replay {replay}", flush=True)
        out.zero_()
        torch.cuda.synchronize()
        graph.launch(s)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), want)


def test_threads_on_one_stream():
    """Calls of several sizes from four threads on one stream keep to their own points."""
    import torch

    mesh = TriMesh(*scenes.noisy_icosphere(5, 1))
    sizes = (17000, 33000, 70000, 150000)
    clouds = [cloud(n, n) for n in sizes]
    want = [mesh.project_local_points(p, True).view(torch.int32).clone() for p in clouds]
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    got, errors = [[] for _ in sizes], []

    def work(k):
        try:
            outs = [torch.zeros(sizes[k], 5, device="cuda") for _ in range(8)]
            torch.cuda.synchronize()
            for o in outs:
                got[k].append(mesh.project_local_points(clouds[k], True, out=o, stream=s))
        except Exception as e:  # reported below
            errors.append(e)

    print("case: four threads", flush=True)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    assert not errors
    for k in range(len(sizes)):
        assert len(got[k]) == 8
        for g in got[k]:
            assert torch.equal(g.view(torch.int32), want[k])


def test_more_points_than_one_sort():
    """2^22 + 20,000 points: the records around the second part's first point, and at both ends, are a small call's."""
    import torch

    mesh = TriMesh(*scenes.noisy_icosphere(3, 1))
    n, part = (1 << 22) + 20000, 1 << 22
    p = cloud(n, 5)
    print(f"case: {n} points", flush=True)
    got = mesh.project_local_points(p, False).view(torch.int32)
    for at in (0, part - 3000, part, n - 3000):
        want = mesh.project_local_points(p[at:at + 3000].contiguous(), False).view(torch.int32)
        assert torch.equal(got[at:at + 3000], want)
