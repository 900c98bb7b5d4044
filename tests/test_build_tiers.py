"""Structure builds at the edges of the build's tiers: one and two
primitives, the largest subtree of a bottom workgroup (256), the largest
count of a one-workgroup build (8,192) and of the middle tier (65,536), each
beside its neighbours; equal Morton codes, skewed trees, signed zeros and NaN
vertices. The blobs equal the oracle's byte for byte."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle_host as oh
from rtg import abi, scenes
from rtg.device import DeviceScene, device_to_host
from rtg.frames import FrameDriver
from rtg.lib import check, load

pytestmark = pytest.mark.gpu


def triangles(kind, n):
    """(n, 3, 3) float32 vertices."""
    rng = scenes.Rng(1000 + n)
    if kind == "same":  # one centre: every Morton code equal
        return np.tile(np.array([[[0, 0, 0], [1, 0, 0], [0, 1, 0]]], np.float32), (n, 1, 1))
    v = scenes.soup(n, 0.02, rng=rng).positions.reshape(n, 3, 3).copy()
    if kind == "skewed":  # sizes and places growing without end: unbalanced treelets
        k = np.arange(n, dtype=np.float64) * (60.0 / n)
        v = (v * (2.0 ** k)[:, None, None]).astype(np.float32)
    elif kind == "flat":  # planes at +0 and -0: ties of box planes
        v[..., 1] = np.where(np.arange(n)[:, None] % 2 == 0, 0.0, -0.0)
    elif kind == "nan":
        v[:: max(2, n // 7), 0, 1] = np.nan
        v[1:: max(3, n // 5), 2, 0] = np.inf
    return v


def gpu_blob(ctx, v, flags):
    n = len(v)
    pos = torch.from_numpy(np.ascontiguousarray(v.reshape(-1, 3))).to("cuda:0")
    idx = torch.arange(3 * n, dtype=torch.int32, device="cuda:0")
    g = abi.Geometry(pos.data_ptr(), 12, 3 * n - 1, idx.data_ptr(), 3 * n, abi.RTG_GEOMETRY_OPAQUE)
    out = C.c_uint64()
    torch.cuda.synchronize()
    check(load().rtg_blas_build(ctx.ptr, C.byref(g), 1, flags, C.byref(out), None), "rtg_blas_build")
    b = device_to_host(out.value, ctx.as_info(out.value).size_bytes)
    check(load().rtg_blas_destroy(ctx.ptr, out.value), "rtg_blas_destroy")
    return b


def oracle_blob(v, flags):
    pos = np.ascontiguousarray(v.reshape(-1, 3))
    idx = np.arange(3 * len(v), dtype=np.uint32)
    g = abi.Geometry(pos.ctypes.data, 12, len(pos) - 1, idx.ctypes.data, len(idx), abi.RTG_GEOMETRY_OPAQUE)
    p, size = C.c_void_p(), C.c_uint64()
    assert oh.lib().orc_blas_build(C.addressof(g), 1, flags, C.byref(p), C.byref(size)) == 0
    b = np.frombuffer(C.string_at(p.value, size.value), dtype=np.uint8).copy()
    oh.lib().orc_free(p)
    return b


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("kind,n", [
    ("soup", 1), ("soup", 2), ("soup", 3), ("soup", 7), ("soup", 8), ("soup", 63), ("soup", 255), ("soup", 256),
    ("soup", 257), ("soup", 1025), ("soup", 8191), ("soup", 8192), ("soup", 8193), ("soup", 65536), ("soup", 65537),
    ("soup", 150001), ("same", 2), ("same", 300), ("same", 9000), ("skewed", 200), ("skewed", 3000),
    ("skewed", 20000), ("flat", 500), ("flat", 10000), ("nan", 40), ("nan", 700), ("nan", 9001)])
def test_blas_bytes_equal_the_oracle(ctx, kind, n, fast):
    v = triangles(kind, n)
    flags = abi.RTG_BUILD_PREFER_FAST_TRACE if fast else 0
    g, o = gpu_blob(ctx, v, flags), oracle_blob(v, flags)
    assert g.shape == o.shape
    assert np.array_equal(g, o)


def test_nine_geometries(ctx):
    """More geometries than a launch carries descriptors of: their flags and
    indices come back in the records."""
    v = triangles("soup", 90)
    pos = torch.from_numpy(np.ascontiguousarray(v.reshape(-1, 3))).to("cuda:0")
    idx = torch.arange(270, dtype=torch.int32, device="cuda:0")
    hp = np.ascontiguousarray(v.reshape(-1, 3))
    hi = np.arange(270, dtype=np.uint32)
    for count in (8, 9, 30):
        gg, og = (abi.Geometry * count)(), (abi.Geometry * count)()
        for k in range(count):
            a, b = 90 * k // count, 90 * (k + 1) // count
            f = abi.RTG_GEOMETRY_OPAQUE if k % 2 else 0
            gg[k] = abi.Geometry(pos.data_ptr(), 12, 269, idx.data_ptr() + 12 * a, 3 * (b - a), f)
            og[k] = abi.Geometry(hp.ctypes.data, 12, 269, hi.ctypes.data + 12 * a, 3 * (b - a), f)
        out = C.c_uint64()
        torch.cuda.synchronize()
        check(load().rtg_blas_build(ctx.ptr, C.cast(gg, C.c_void_p), count, abi.RTG_BUILD_PREFER_FAST_TRACE,
                                    C.byref(out), None), "rtg_blas_build")
        g = device_to_host(out.value, ctx.as_info(out.value).size_bytes)
        check(load().rtg_blas_destroy(ctx.ptr, out.value), "rtg_blas_destroy")
        p, size = C.c_void_p(), C.c_uint64()
        assert oh.lib().orc_blas_build(C.addressof(og), count, abi.RTG_BUILD_PREFER_FAST_TRACE, C.byref(p),
                                       C.byref(size)) == 0
        o = np.frombuffer(C.string_at(p.value, size.value), dtype=np.uint8).copy()
        oh.lib().orc_free(p)
        assert np.array_equal(g, o)


def _masked(blob, n):
    """TLAS blob bytes without the BLAS addresses (device or host pointers)."""
    b = np.frombuffer(blob, dtype=np.uint8).copy()
    hdr = b[:128].view(np.uint64)
    for off, at in ((int(hdr[9]), 48), (int(hdr[10]), 56)):
        b[off:off + 64 * n].reshape(n, 64)[:, at:at + 8] = 0
    return b


@pytest.mark.parametrize("n", [1, 2, 256, 257, 1500, 5003, 8192, 8193, 20011])
def test_tlas_bytes_and_refit_equal_the_oracle(ctx, n):
    """The build, and the update whose launches go by the levels' sizes: of a
    clone, of the structure itself, and of a frame slot's copy."""
    rng = scenes.Rng(7 + n)
    s = scenes.Scene("crowd")
    s.add_mesh(scenes.icosphere(1))
    s.add_mesh(scenes.quad(2.0, 1.0))
    s.models.append(scenes.Model(0, [(0, 0, -1)]))
    scenes._base_textures(s, 7)
    side = np.sqrt(n)
    p = rng.uniform(3 * n, -side, side).reshape(n, 3)
    for k in range(n):
        s.instances.append(scenes.InstanceData(scenes.affine(p[k], None, 0.7), 0, k % 2))
    ds, hs = DeviceScene(ctx, s), oh.HostScene(s)
    assert np.array_equal(_masked(ds.as_bytes(ds.tlas), n), _masked(hs.tlas.bytes(), n))
    turn = rng.uniform(3 * n).reshape(n, 3)
    step = rng.uniform(3 * n, -1.0, 1.0).reshape(n, 3)
    xf = [scenes.affine(p[k] + step[k], scenes.rotation_from_uniform(*turn[k]), 0.9) for k in range(n)]
    clone, buf = ds.clone_tlas(), ds.instance_buffer(xf)
    torch.cuda.synchronize()
    hs.refit(xf)
    want = _masked(hs.tlas.bytes(), n)
    for tlas in (clone, ds.tlas):
        ds.refit(buf, tlas=tlas)
        torch.cuda.synchronize()
        assert np.array_equal(_masked(ds.as_bytes(tlas), n), want)
    driver = FrameDriver(ds, 1)
    inst, slot = driver.begin(0)
    inst["transform"] = np.asarray(xf, np.float32)
    s.width = s.height = 8
    out = ds.make_outputs()
    driver.submit(0, ds.job(out))
    torch.cuda.synchronize()
    assert np.array_equal(_masked(ds.as_bytes(slot), n), want)
    driver.close()
    check(load().rtg_tlas_destroy(ctx.ptr, clone), "rtg_tlas_destroy")
    ds.destroy()
