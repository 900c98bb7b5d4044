"""Traces in flight together: a trace enqueued while another stream's is on the
GPU runs its bounce levels in sequence, alone it runs them beside the first
level's shadow rays. The images are the same bit for bit, and a frame alone
equals the oracle's."""
import numpy as np
import pytest
import torch

import oracle_host as oh
from rtg import scenes
from rtg.device import DeviceScene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (33, 17), (320, 180), (400, 300)])
@pytest.mark.parametrize("streams", [1, 3])
def test_images_do_not_depend_on_what_is_in_flight(ctx, w, h, streams):
    s = scenes.default_scene(n_tori=12, width=w, height=h)
    s.shadow_rays = 3
    ds = DeviceScene(ctx, s)
    alone = [ds.trace_image(frame_index=f) for f in range(2)]
    torch.cuda.synchronize()
    o_rgba, o_rgb, _, _ = oh.HostScene(s).trace_image(frame_index=0)
    assert np.array_equal(alone[0][0].cpu().numpy().view(np.uint32), o_rgba)
    ss = [torch.cuda.Stream() for _ in range(streams)]
    outs = []
    for k in range(8):
        with torch.cuda.stream(ss[k % streams]):
            outs.append(ds.trace_image(frame_index=k % 2))
    torch.cuda.synchronize()
    for k, out in enumerate(outs):
        for got, want in zip(out[:2], alone[k % 2][:2]):
            assert torch.equal(got.view(torch.int32), want.view(torch.int32)), k
    ds.destroy()
