"""Small calls of the static and binned ray mappings put fewer rays in a wave: at the
sizes where their number changes, the hits and node counts are those of a call large
enough for full waves (cast_local_ray_and_get_normal, ray_trimesh.rs:12-130)."""
import numpy as np
import pytest

from parry_amd import TriMesh, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mapping,block", [("static", 256), ("static", 64), ("binned", 128)])
@pytest.mark.parametrize("level", [0, 4])
def test_few_rays_per_wave(mapping, block, level):
    import torch

    v, f = scenes.noisy_icosphere(level, 1)
    mesh = TriMesh(v, f)
    many = scenes.rays_into_unit_ball(70000, 2)
    many[::7, 4] = 0.0  # waves with and without a zero direction component
    rays = torch.from_numpy(many).cuda()
    mesh.set_tuning("static")
    want = mesh.cast_local_rays_and_get_normal(rays, 10.0, True).view(torch.int32)
    culled = mesh.cast_local_rays_with_culling(rays, 10.0, "ignore_backfaces").view(torch.int32)
    mesh.set_tuning(mapping, block_size=block)
    for n in (1, 2, 3, 63, 1023, 1024, 1025, 8192, 8193, 20480, 20481, 32768, 32769, 65536, 65537):
        print(f"case: {mapping} {block}, level {level}, {n} rays", flush=True)
        got = mesh.cast_local_rays_and_get_normal(rays[:n].contiguous(), 10.0, True).view(torch.int32)
        assert torch.equal(got, want[:n])
        got = mesh.cast_local_rays_with_culling(rays[:n].contiguous(), 10.0, "ignore_backfaces").view(torch.int32)
        assert torch.equal(got, culled[:n])
    assert np.isfinite(want.view(torch.float32).cpu().numpy()[:, 0]).any()
