"""Closest-hit queries of more rays than four workgroups per CU hold (262,144),
which run on five with 15 stack entries a lane in LDS: sizes at the edges of
both grids equal the oracle's hits bit for bit, and stacks past the 15th entry
equal the counted query's, which keeps four workgroups and 16 entries."""
import numpy as np
import pytest
import torch

import oracle_host as oh
from rtg import abi, scenes
from rtg.device import DeviceScene, hits_to_numpy, rays_to_device

pytestmark = pytest.mark.gpu


def _hits(ds, rays):
    out = ds.trace_rays(rays_to_device(rays), len(rays))
    torch.cuda.synchronize()
    return hits_to_numpy(out).view(np.uint32)


@pytest.mark.parametrize("n", [262144, 262145, 327680, 327681, 400003])
def test_sizes(ctx, n):
    s = scenes.default_scene(n_tori=20, width=64, height=48)
    ds = DeviceScene(ctx, s)
    rays = scenes.incoherent_rays(n, (-10, 0, -10), (10, 3, 10), seed=n)
    ref, _ = oh.HostScene(s).trace_rays(rays)
    assert np.array_equal(_hits(ds, rays), ref.view(np.uint32))
    ds.destroy()


def test_stacks_past_their_lds_part(ctx):
    """Rays that overlap every box of a 4,096-instance TLAS, all but every 64th
    instance masked, of one small triangle."""
    rng = scenes.Rng(9)
    v = np.array([[-1.0, -0.9, -1.1], [1.1, 1.0, -0.9], [-0.9, 1.1, 1.0]], dtype=np.float32)
    m = scenes.Mesh("one", v, np.tile([[0.0, 1.0, 0.0]], (3, 1)), np.zeros((3, 2)), [(np.arange(3).reshape(1, 3), True)])
    s = scenes.Scene("deep")
    scenes._base_textures(s, 7)
    s.add_mesh(m)
    s.add_model(0, [s.material((0.5, 0.5, 0.5), 0.5)])
    p = rng.uniform(3 * 4096, -0.05, 0.05).reshape(4096, 3)
    for k in range(4096):
        s.instances.append(scenes.InstanceData(scenes.affine(p[k]), 0, 0, mask=0xFF if k % 64 == 0 else 0))
    s.width, s.height = 4, 4
    s.view_inverse = scenes.look_at_inverse((0.0, 0.1, 3.0), (0.0, 0.0, 0.0))
    s.proj_inverse = scenes.proj_inverse_reversed_z(0.6, 1.0)
    s.sun_dir = scenes.sun_direction(0.6, 0.4)
    ds = DeviceScene(ctx, s)
    rays = scenes.incoherent_rays(270001, (-0.5, -0.5, -0.5), (0.5, 0.5, 0.5), seed=4)
    got = _hits(ds, rays)
    ctx.set_counters(True)
    try:
        want = _hits(ds, rays)
        deep = ctx.counters().spill_pushes
    finally:
        ctx.set_counters(False)
    assert deep > 0
    assert np.array_equal(got, want)
    ds.destroy()
