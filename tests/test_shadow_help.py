"""The bounce stream's workgroups trace first-level shadow rays once the bounce
levels are done, where the launch beside them has more pairs than lanes: with
bounce shadow rays traced by four lanes a pair and by one, and few or many
workgroups on the bounce stream. Images equal the oracle's bit for bit."""
import numpy as np
import pytest
import torch

import oracle_host as oh
from rtg import abi, scenes
from rtg.device import DeviceScene, hits_to_numpy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bounce_blocks", [1, 3, 8, 64, 4096])
@pytest.mark.parametrize("mirror_floor", [False, True])
@pytest.mark.parametrize("shadow_rays", [1, 3])
def test_first_level_pairs_beyond_the_grid(ctx, bounce_blocks, mirror_floor, shadow_rays):
    s = scenes.default_scene(width=401, height=299, n_tori=30)
    if mirror_floor:
        s.instances[0].hit_group = abi.RTG_HIT_MIRROR
    ds, hs = DeviceScene(ctx, s), oh.HostScene(s)
    o = s.trace_opts()
    o.shadow_rays = shadow_rays
    saved = ctx.tuning()
    ctx.set_tuning(abi.Tuning.make(**{**saved.as_dict(), "blocks_per_cu": 1, "bounce_blocks": bounce_blocks}))
    try:
        outs = []
        for _ in range(3):
            outs.append(ds.trace_image(frame_index=3, opts=o))
            torch.cuda.synchronize()
    finally:
        ctx.set_tuning(saved)
    o_rgba, o_rgb, o_hits, oc = hs.trace_image(frame_index=3, opts=o)
    if mirror_floor:
        assert oc.bounce_rays > 16384
    for rgba, rgb, ph in outs:
        assert np.array_equal(hits_to_numpy(ph).view(np.uint32), o_hits.view(np.uint32))
        assert np.array_equal(rgba.cpu().numpy().view(np.uint32), o_rgba)
    ds.destroy()
