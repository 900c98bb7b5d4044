"""Structures built into the memory of destroyed ones: the blobs equal the
oracle's byte for byte whatever the block held, and a context keeps at most
128 MiB of destroyed structures."""
import numpy as np
import pytest
import torch

from rtg import abi
from rtg.lib import Context
from test_build_tiers import gpu_blob, oracle_blob, triangles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(500, 450, 500, 401, 1), (9000, 8191, 8500, 7001, 9000), (2, 3, 2, 1, 2)])
def test_blobs_in_reused_memory(ctx, sizes):
    for k, n in enumerate(sizes):
        v = triangles("soup", n) + np.float32(k)
        flags = abi.RTG_BUILD_PREFER_FAST_TRACE if k % 2 else 0
        assert np.array_equal(gpu_blob(ctx, v, flags), oracle_blob(v, flags))


def test_destroyed_structures_are_bounded_and_given_back():
    c = Context(0)
    v = [triangles("soup", n) for n in (200_000, 260_000, 340_000, 440_000, 600_000)]
    gpu_blob(c, v[-1], 0)  # the build's scratch at its largest
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    for a in v * 2:
        gpu_blob(c, a, 0)
        torch.cuda.empty_cache()
        assert before - torch.cuda.mem_get_info()[0] <= (128 << 20) + (8 << 20)
    c.close()
    assert torch.cuda.mem_get_info()[0] >= before


def test_a_block_beyond_the_bound_leaves_the_kept_ones():
    """A structure of more than 128 MiB is never kept; destroying it leaves
    what the context keeps of smaller ones."""
    c = Context(0)
    rng = np.random.default_rng(3)
    large, small = (rng.random((n, 3, 3), dtype=np.float32) for n in (2_000_000, 1_000_000))
    assert len(gpu_blob(c, large, 0)) > 128 << 20  # and the build's scratch at its largest
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    kept = len(gpu_blob(c, small, 0))
    gpu_blob(c, large, 0)
    torch.cuda.empty_cache()
    assert before - torch.cuda.mem_get_info()[0] >= kept
    c.close()
