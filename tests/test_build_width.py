"""Builds with treelets on both sides of the size up to which a bottom
subtree takes 512 lanes (80,000 primitives); beyond it takes 256. Builds at
the edges of the sort's tiles (2,048 keys) and of the count up to which its
scatter sums the tiles itself (262,144). The blobs equal the oracle's byte for
byte."""
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


@pytest.mark.parametrize("kind", ["soup", "same"])
@pytest.mark.parametrize("n", [8193, 10239, 10240, 10241, 262144, 262145])
def test_sorted_orders(ctx, kind, n):
    v = triangles(kind, n)
    assert np.array_equal(gpu_blob(ctx, v, 0), oracle_blob(v, 0))
