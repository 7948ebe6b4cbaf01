"""Scenes 1e8 units and more across against the oracle's linear scan: rays with a
direction component that is exactly zero must keep their hits whatever the
products of a walk come to (the 4-wide nodes in LDS, in memory and in their
half-size form, and the wavefront's kernels)."""
import numpy as np
import pytest

import oracle
import raydar_amd as ra
from raydar_amd import abi, scene, scenegen

pytestmark = pytest.mark.gpu


def _mirrors(objects, power, side, size=1.0):
    # An orthographic camera along z: a camera ray's direction points from its
    # pixel's place to 0 (cpu.rs:234-251), so the column at a quarter of the
    # width holds rays in the plane x = 8 with no x component, the row at three
    # quarters of the height such rays in y = 8, and mirror cubes send them on.
    s = 2.0 ** power
    sc = scenegen.clustered(6, objects, side, side)
    sc.objects["kind"][::2] = abi.RD_CUBE
    sc.objects["metallic"][::2] = 1.0
    sc.objects["roughness"][::2] = 0.0
    sc.objects["transmission"][::2] = 0.0
    sc.objects["center"][::8, 0] = sc.objects["center"][4::8, 1] = 8.0
    sc.objects["center"] *= np.float32(s)
    sc.objects["size"] *= np.float32(s * size)
    sc.camera = scene.make_camera((8 * s, 8 * s, -64 * s), (8 * s, 8 * s, 0), (0, 1, 0), side, side,
                                  ortho_size=16 * s, near=0.1 * s, far=200 * s)
    y, x = np.mgrid[:side, :side]
    lines = (x == side // 4) | (x == 3 * side // 4) | (y == side // 4) | (y == 3 * side // 4)
    pix = np.flatnonzero(lines | ((x + 31 * y) % 1999 == 0)).astype(np.uint32)
    rays = oracle.camera_rays(sc, pix)
    hit = oracle.trace(sc, rays)[0] >= 0
    assert (hit & (rays[:, 3] == 0)).sum() > 20 and (hit & (rays[:, 4] == 0)).sum() > 20
    return sc, pix


@pytest.mark.parametrize("power", [24, 25, 26, 28, 40])
def test_half_size_nodes_keep_axis_parallel_hits(power):
    # 14000 objects and enough paths for the half-size form
    sc, pix = _mirrors(14000, power, 1536)
    print(f"half-size nodes, scale 2^{power}", flush=True)
    with ra.HipRenderer(max_sample_count=2, max_bounces=4, seed=3) as r:
        r.render_frame(sc)
        acc = r.accumulator()
    ref = oracle.render(sc, 2, 4, 3, pixels=pix, threads=8)
    np.testing.assert_array_equal(acc[pix].view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("opts", [dict(), dict(lds_bvh=0), dict(block=128), dict(refill=0), dict(bvh4=0)])
@pytest.mark.parametrize("power", [26, 28, 40])
def test_trees_keep_axis_parallel_hits(power, opts):
    sc, pix = _mirrors(120, power, 128, 4.0)
    print(f"trees, scale 2^{power}, {opts}", flush=True)
    with ra.HipRenderer(max_sample_count=3, max_bounces=8, seed=3, **opts) as r:
        r.render_frame(sc)
        acc = r.accumulator()
    ref = oracle.render(sc, 3, 8, 3)
    np.testing.assert_array_equal(acc.view(np.uint32), ref.view(np.uint32))
