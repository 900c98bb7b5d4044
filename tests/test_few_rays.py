"""Launches of few rays, which take four lanes a ray: at the edges of a wave,
of a workgroup and of the default grid's capacity (65,536), with stacks past
their LDS part, in images and bounce levels on both sides of the capacity.
Hits, occlusion and images equal the oracle's bit for bit."""
import numpy as np
import pytest
import torch

import oracle_host as oh
from rtg import abi, scenes
from rtg.device import DeviceScene, hits_to_numpy, rays_to_device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fences(ctx):
    s = scenes.default_scene(n_tori=20, width=64, height=48)
    ds = DeviceScene(ctx, s)
    yield s, ds, oh.HostScene(s)
    ds.destroy()


def _same_rays(ds, hs, rays, mode, **kw):
    out = ds.trace_rays(rays_to_device(rays), len(rays), mode=mode, **kw)
    torch.cuda.synchronize()
    ref, _ = hs.trace_rays(rays, mode=mode, **kw)
    got = hits_to_numpy(out) if mode == abi.RTG_QUERY_CLOSEST else out.cpu().numpy()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    return ref


@pytest.mark.parametrize("n", [1, 3, 4, 5, 16, 17, 63, 64, 65, 4095, 4096, 4097, 65535, 65536, 65537])
@pytest.mark.parametrize("mode", [abi.RTG_QUERY_CLOSEST, abi.RTG_QUERY_OCCLUSION])
def test_query_sizes(ctx, fences, n, mode):
    s, ds, hs = fences
    rays = scenes.incoherent_rays(n, (-10, 0, -10), (10, 3, 10), seed=50 + n)
    _same_rays(ds, hs, rays, mode)


@pytest.mark.parametrize("flags,mask,sbt", [(0, 0xFF, 1), (abi.RTG_RAY_FLAG_OPAQUE, 0xFF, 0),
                                            (abi.RTG_RAY_FLAG_NO_OPAQUE, 0xFF, 0),
                                            (abi.RTG_RAY_FLAG_TERMINATE_ON_FIRST_HIT, 0xFF, 0), (0, 0x00, 0)])
def test_query_flags(ctx, fences, flags, mask, sbt):
    s, ds, hs = fences
    rays = scenes.incoherent_rays(3000, (-10, 0, -10), (10, 3, 10), seed=3)
    for mode in (abi.RTG_QUERY_CLOSEST, abi.RTG_QUERY_OCCLUSION):
        _same_rays(ds, hs, rays, mode, ray_flags=flags, cull_mask=mask, sbt_offset=sbt)


@pytest.mark.parametrize("entries", [8, 16])
def test_stacks_past_their_lds_part(ctx, entries):
    """Rays that overlap every box of a 4,096-instance TLAS (all but every
    64th instance masked) and of a 1,024-triangle BLAS."""
    rng = scenes.Rng(5)
    n = 1024
    c = rng.uniform(3 * n, -0.05, 0.05).reshape(n, 1, 3)
    v = (c + np.array([[-1.0, -0.9, -1.1], [1.1, 1.0, -0.9], [-0.9, 1.1, 1.0]])).astype(np.float32)
    m = scenes.Mesh("overlapping", v.reshape(-1, 3), np.tile([[0.0, 1.0, 0.0]], (3 * n, 1)), np.zeros((3 * n, 2)),
                    [(np.arange(3 * n).reshape(-1, 3), True)])
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
    s.shadow_rays = 3
    ds, hs = DeviceScene(ctx, s), oh.HostScene(s)
    saved = ctx.tuning()
    ctx.set_tuning(abi.Tuning.make(**{**saved.as_dict(), "stack_lds_entries": entries}))
    try:
        rays = scenes.incoherent_rays(9, (-0.2, -0.2, -0.2), (0.2, 0.2, 0.2), seed=4)
        ctx.set_counters(True)
        ds.trace_rays(rays_to_device(rays), 9)
        deep = ctx.counters().spill_pushes
        ctx.set_counters(False)
        assert deep > 0  # past 16 entries a lane, the counted kernel says
        for mode in (abi.RTG_QUERY_CLOSEST, abi.RTG_QUERY_OCCLUSION):
            _same_rays(ds, hs, rays, mode)
        rgba, rgb, ph = ds.trace_image()
        torch.cuda.synchronize()
        o_rgba, o_rgb, o_hits, _ = hs.trace_image()
        assert np.array_equal(hits_to_numpy(ph).view(np.uint32), o_hits.view(np.uint32))
        assert np.array_equal(rgba.cpu().numpy().view(np.uint32), o_rgba)
    finally:
        ctx.set_counters(False)
        ctx.set_tuning(saved)
        ds.destroy()


@pytest.mark.parametrize("w,h,spp,shadow_rays,bounce_blocks", [
    (5, 3, 1, 2, 192), (16, 16, 1, 1, 192), (256, 256, 1, 2, 192), (257, 256, 1, 2, 192), (128, 128, 4, 3, 8),
    (96, 80, 2, 4, 0), (96, 80, 2, 4, 3), (400, 300, 1, 2, 192), (400, 300, 1, 2, 0)])
def test_images_and_bounce_levels(ctx, w, h, spp, shadow_rays, bounce_blocks):
    """A mirror floor, so that the larger images' bounce levels hold more rays
    than the capacity and the smaller ones' fewer."""
    s = scenes.default_scene(width=w, height=h, n_tori=30)
    s.instances[0].hit_group = abi.RTG_HIT_MIRROR
    ds, hs = DeviceScene(ctx, s), oh.HostScene(s)
    o = s.trace_opts()
    o.spp, o.shadow_rays = spp, shadow_rays
    saved = ctx.tuning()
    ctx.set_tuning(abi.Tuning.make(**{**saved.as_dict(), "bounce_blocks": bounce_blocks}))
    try:
        rgba, rgb, ph = ds.trace_image(frame_index=3, opts=o)
        torch.cuda.synchronize()
    finally:
        ctx.set_tuning(saved)
    o_rgba, o_rgb, o_hits, oc = hs.trace_image(frame_index=3, opts=o)
    if w * h * spp > 100_000:
        assert oc.bounce_rays > 65536
    assert np.array_equal(hits_to_numpy(ph).view(np.uint32), o_hits.view(np.uint32))
    assert np.array_equal(rgba.cpu().numpy().view(np.uint32), o_rgba)
    assert float(np.abs(rgb.cpu().numpy().reshape(-1, 3) - o_rgb).max()) <= 1e-4
    ds.destroy()
