"""Streams that the library makes for itself and destroys (a batch's capture,
the autotuner's runs) leave nothing behind that still refers to them: HIP asks
an event's stream whether it is being captured, so an event that outlives its
stream answers for whatever stream takes that memory next. Here those are
streams under capture."""
import contextlib
import ctypes

import pytest
import torch

from rtg import scenes
from rtg.batch import Batch, autotune
from rtg.device import DeviceScene

pytestmark = pytest.mark.gpu

RELAXED = 2  # hipStreamCaptureModeRelaxed: other work of the thread goes on


@contextlib.contextmanager
def streams_under_capture(count):
    hip = ctypes.CDLL("libamdhip64.so")
    streams = [ctypes.c_void_p() for _ in range(count)]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0  # non-blocking
        assert hip.hipStreamBeginCapture(s, RELAXED) == 0
    try:
        yield
    finally:
        ended = []
        for s in streams:
            g = ctypes.c_void_p()
            ended.append(hip.hipStreamEndCapture(s, ctypes.byref(g)))
            if g.value:
                hip.hipGraphDestroy(g)
            hip.hipStreamDestroy(s)
    assert ended == [0] * count
    assert hip.hipGetLastError() == 0


@pytest.fixture
def scene(ctx):
    ds = DeviceScene(ctx, scenes.default_scene(n_tori=5, width=64, height=48))
    alone = ds.trace_image(frame_index=1)[0]
    torch.cuda.synchronize()
    yield ds, alone.clone()
    ds.destroy()


@pytest.mark.parametrize("count", [1, 4, 16])
def test_batch_updated_while_streams_are_captured(ctx, scene, count):
    ds, alone = scene
    out = ds.make_outputs(hits=False)
    stream = torch.cuda.Stream()
    for _ in range(4):
        b = Batch(ctx, [ds.job(out, frame_index=0)])
        with streams_under_capture(count):
            b.update([ds.job(out, frame_index=1)], stream=stream)
        b.launch(stream)
        torch.cuda.synchronize()
        assert torch.equal(out[0], alone)
        b.close()


@pytest.mark.parametrize("count", [1, 4, 16])
def test_trace_after_tuning_while_streams_are_captured(ctx, scene, count):
    ds, alone = scene
    out = ds.make_outputs(hits=False)
    saved = ctx.tuning()
    try:
        autotune(ctx, [ds.job(out, frame_index=0)], repeats=1)
    finally:
        ctx.set_tuning(saved)
    with streams_under_capture(count):
        got = ds.trace_image(frame_index=1)[0]
    torch.cuda.synchronize()
    assert torch.equal(got, alone)
