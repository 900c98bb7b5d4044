"""The slots that a workgroup takes from the frame's queues, round after round,
whatever order its waves run in: csrc/queue_alloc.hpp on the CPU, a fiber per
lane, under every order of priority of the four waves. On the GPU, an image of
more paths than two rounds of its shading launch hold, with workgroups that
are empty in the last round, against the oracle."""
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG, REPO


def test_slots_under_every_order_of_the_waves(tmp_path):
    exe = str(tmp_path / "queue_alloc_sim")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(PKG, "csrc"), "-o", exe,
                    os.path.join(REPO, "tests", "queue_alloc_sim.cpp")], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert "queue slots: ok" in r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("njobs", [1, 2])
def test_images_of_several_rounds(ctx, njobs):
    """2.19 M paths: two full rounds of 4,096 workgroups and a part of a third;
    63,918 bounce rays, more than the bounce levels' 192 workgroups hold."""
    import torch

    import oracle_host as oh
    from rtg import scenes
    from rtg.batch import trace_batch
    from rtg.device import DeviceScene

    s = scenes.default_scene(n_tori=12, width=1993, height=1101)
    assert s.width * s.height > 2 * 256 * 16 * 256
    ds, hs = DeviceScene(ctx, s), oh.HostScene(s)
    want = []
    for f in range(njobs):
        rgba, _, _, cnt = hs.trace_image(frame_index=f, want_hits=False)
        assert cnt.bounce_rays > 192 * 256
        want.append(rgba)
    for _ in range(3):
        outs = [ds.make_outputs(hits=False) for _ in range(njobs)]
        trace_batch(ctx, [ds.job(o, frame_index=f) for f, o in enumerate(outs)])
        torch.cuda.synchronize()
        for f, o in enumerate(outs):
            assert np.array_equal(o[0].cpu().numpy().view(np.uint32), want[f]), f
    ds.destroy()
