"""Builds with treelets on both sides of the size up to which a bottom
subtree takes 512 lanes (80,000 primitives); beyond it takes 256. The blobs
equal the oracle's byte for byte."""
import numpy as np
import pytest

from rtg import abi
from test_build_tiers import gpu_blob, oracle_blob, triangles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["soup", "flat", "nan", "skewed"])
@pytest.mark.parametrize("n", [70000, 80000, 80001])
def test_blas_bytes_equal_the_oracle(ctx, kind, n):
    v = triangles(kind, n)
    flags = abi.RTG_BUILD_PREFER_FAST_TRACE
    assert np.array_equal(gpu_blob(ctx, v, flags), oracle_blob(v, flags))
