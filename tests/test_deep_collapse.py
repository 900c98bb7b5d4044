"""Builds whose collapse takes more turns than one: a broad level of more wide
nodes than the first workgroup takes (2,048) and more levels below it than are
launched between two looks at the progress (12, and twice that). The blobs
equal the oracle's byte for byte."""
import numpy as np
import pytest

from rtg import abi
from test_build_tiers import gpu_blob, oracle_blob

pytestmark = pytest.mark.gpu


def deep_below_broad(n_broad, chains, steps):
    """(n, 3, 3) vertices: a uniform cloud of small triangles, and under
    corners of its grid of Morton cells a chain of ever closer groups of four,
    each larger than all that follows. A wide node opens the group, so the
    chain gives a level for each of its steps."""
    rng = np.random.default_rng(5)
    c = rng.random((n_broad, 3))
    c[:2] = [[0, 0, 0], [1, 1, 1]]  # the bounds of the centres
    v = [c[:, None, :] + rng.normal(0, 1e-3, (n_broad, 3, 3)) * np.array([1, 0, 0])[None, :, None]]
    v[0][:, 2] = 2 * c - v[0][:, 1]  # boxes centred on c
    v[0][:, 0] = c
    for k in range(chains):
        at = (np.array([(k * 7) % 16, (k * 3) % 16, (k * 11) % 16]) * 64 + 0.5) / 1024
        for j in range(30 - steps, 30):
            g = at.copy()
            g[j % 3] += 2.0 ** (9 - j // 3) / 1024
            s = 0.5 * 0.8 ** (j + steps - 30)
            v.append(np.tile(np.stack([g - s / 2, g + s / 2, g])[None], (4, 1, 1)))
        v.append(np.tile(np.stack([at - 1e-3, at + 1e-3, at])[None], (4096 if k == 0 else 40, 1, 1)))
    return np.concatenate(v).astype(np.float32)


def level_sizes(blob):
    """Nodes of each breadth-first level of a blob (numbered level by level)."""
    header = blob[:128]
    n, off = int(header.view(np.uint32)[2]), int(header.view(np.uint64)[8])
    child = blob[off:off + 128 * n].view(np.uint32).reshape(n, 32)[:, 24:28]
    inner = (child & np.uint32(0x80000000)) == 0  # an empty slot has the leaf bit
    sizes, first = [], 0
    while first < n:
        end = first + (sizes[-1] if sizes else 1)
        sizes.append(int(inner[first:end].sum()))
        first = end
    return [1] + sizes[:-1]



@pytest.mark.parametrize("n_broad,chains,steps,turns", [(9000, 1, 18, 3), (20000, 2, 8, 2), (150000, 9, 18, 3)])
@pytest.mark.parametrize("flags", [0, abi.RTG_BUILD_PREFER_FAST_TRACE])
def test_blas_bytes_equal_the_oracle(ctx, n_broad, chains, steps, turns, flags):
    v = deep_below_broad(n_broad, chains, steps)
    want = oracle_blob(v, flags)
    sizes = level_sizes(want)
    broad = next(k for k, m in enumerate(sizes) if m > 2048)
    assert 12 * (turns - 1) < len(sizes) - broad  # the broad level is the first of the first turn
    got = gpu_blob(ctx, v, flags)
    assert got.shape == want.shape
    assert np.array_equal(got, want)
