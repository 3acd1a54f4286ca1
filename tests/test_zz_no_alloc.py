"""rgExtTraceRaysNoAlloc, the allocation-free variant of rgExtTraceRays,
against rgExtTraceRays through the C ABI: the same hits bit for bit (t, u,
v, primitive id), the same node / triangle counts and no error bits, for
closest-hit and any-hit rays, FP32 and FP16 nodes, on two calls in a row
whose second has fewer rays (the shared scratch keeps the last call's
contents and is cleared by every call)."""
import numpy as np
import pytest

from raytracedgl1_amd import ffi, scenes
from raytracedgl1_amd.ffi import HIT_DTYPE, Bvh, DeviceArray

pytestmark = pytest.mark.gpu


def _rays():
    cam = scenes.terrain_boxes_camera()
    big = scenes.primary_rays(cam, 320, 180)
    other = scenes.Camera(cam.eye + np.array([3.0, 1.0, -2.0]), cam.target)
    small = scenes.primary_rays(other, 96, 54)
    return big, small


def _no_alloc(b, d_rays, n, d_hits, flags):
    ffi.call("rgExtTraceRaysNoAlloc", b.h, d_rays.ptr, n, d_hits.ptr, flags, None)


@pytest.mark.parametrize("fmt", [ffi.RG_EXT_BVH_NODE_FP32, ffi.RG_EXT_BVH_NODE_FP16])
def test_no_alloc_trace_equals_trace(gpu, fmt):
    s = scenes.terrain_boxes_scene()
    b = Bvh()
    b.build(DeviceArray.from_numpy(np.ascontiguousarray(s.tris, np.float32)), len(s.tris), 3, fmt)
    big, small = _rays()
    for flags in (0, ffi.RG_EXT_TRACE_ANY_HIT, ffi.RG_EXT_TRACE_COLLECT_STATS,
                  ffi.RG_EXT_TRACE_ANY_HIT | ffi.RG_EXT_TRACE_COLLECT_STATS, ffi.RG_EXT_TRACE_CULL_FRONT_FACE):
        for rays in (big, small):  # the second call has fewer rays
            print(f"no-alloc trace: node format {fmt}, flags {flags}, {len(rays)} rays", flush=True)
            dr = DeviceArray.from_numpy(rays)
            ref = DeviceArray(len(rays), HIT_DTYPE)
            got = DeviceArray(len(rays), HIT_DTYPE)
            b.trace(dr, len(rays), ref, flags)
            want = ref.download()
            want_stats = b.trace_stats() if flags & ffi.RG_EXT_TRACE_COLLECT_STATS else None
            assert b.trace_errors() == 0
            _no_alloc(b, dr, len(rays), got, flags)
            h = got.download()
            assert b.trace_errors() == 0
            for f in ("prim", "t", "u", "v") if flags != ffi.RG_EXT_TRACE_ANY_HIT else ():
                assert np.array_equal(h[f], want[f]), (fmt, flags, len(rays), f)
            assert np.array_equal(h["prim"] == ffi.RG_EXT_MISS, want["prim"] == ffi.RG_EXT_MISS)
            # front-face culling leaves the back faces only
            assert (h["prim"] != ffi.RG_EXT_MISS).mean() > (0.1 if flags & ffi.RG_EXT_TRACE_CULL_FRONT_FACE else 0.5)
            if want_stats is not None:
                assert b.trace_stats() == want_stats


def test_no_alloc_trace_rejects_too_many_rays(gpu):
    s = scenes.terrain_boxes_scene()
    b = Bvh()
    b.build(DeviceArray.from_numpy(np.ascontiguousarray(s.tris, np.float32)), len(s.tris), 3)
    dr = DeviceArray(16, ffi.RAY_DTYPE)
    dh = DeviceArray(16, HIT_DTYPE)
    with pytest.raises(ffi.RgError) as e:
        ffi.call("rgExtTraceRaysNoAlloc", b.h, dr.ptr, 0xF0000001, dh.ptr, 0, None)  # rejected before any launch
    assert e.value.code == ffi.RG_RESULT_WRONG_FUNCTION_ARGUMENT
    _no_alloc(b, dr, 0, dh, 0)  # zero rays: nothing to do
