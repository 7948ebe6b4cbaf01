"""rd_render_frame_noalloc of scenes whose arrays exceed the upload memory that
rd_create reserved (256 KB, 8 MB): they go through it in parts, and the images
are rd_render_frame's."""
import ctypes as C

import numpy as np
import pytest

import raydar_amd as ra
from raydar_amd import abi, scenegen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opts", [dict(), dict(block=128)])
@pytest.mark.parametrize("objects", [1100, 1300, 5000, 60000])
def test_large_scenes_match_render_frame(objects, opts):
    sc = scenegen.clustered(8, objects, 320, 180)
    out = np.zeros((sc.height, sc.width, 4), np.uint8)
    f = ra.lib().rd_render_frame_noalloc
    f.restype, f.argtypes = C.c_int, [C.c_void_p, C.POINTER(abi.RdScene), C.c_void_p, C.c_size_t]
    print(f"noalloc, {objects} objects, {opts}", flush=True)
    with ra.HipRenderer(max_sample_count=3, max_bounces=8, seed=5, **opts) as r:
        want = r.render_frame(sc)
        s = sc.as_rd()
        for _ in range(2):
            ra.check(f(r._h, C.byref(s), out.ctypes.data_as(C.c_void_p), out.nbytes), r._h)
            np.testing.assert_array_equal(out, want)
            out[:] = 0
