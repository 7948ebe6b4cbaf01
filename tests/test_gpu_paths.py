"""The path kernel (paths.hip): one scene's whole paths in one launch.

Frames against the oracle bit for bit (every draw is keyed by pixel, sample
and bounce, so neither the order of the paths nor the lanes that carry them
may show) where its work list and its turns have edges: images of fewer
pixels than a group of 64, groups that are not full, sample counts that do
not divide the slices, one workgroup, turns at 1 to 64 idle lanes, a tree in
LDS or not, leaves of several primitives, one bounce.
"""
import ctypes as C

import numpy as np
import pytest

import oracle
import raydar_amd as ra
from raydar_amd import abi, scene, scenegen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,spp,bounces,opts", [
    ((1, 1), 3, 12, dict()), ((1, 1), 200, 4, dict()), ((7, 9), 5, 12, dict()),
    ((8, 8), 33, 12, dict()), ((65, 1), 32, 12, dict()), ((3, 43), 31, 8, dict()),
    ((64, 64), 2, 1, dict()), ((200, 130), 1, 12, dict()), ((121, 77), 7, 12, dict(grid=1)),
    ((121, 77), 6, 12, dict(refill=1)), ((121, 77), 6, 12, dict(refill=15, grid=3)),
    ((121, 77), 6, 12, dict(refill=16)), ((121, 77), 6, 12, dict(refill=64)),
    ((121, 77), 6, 12, dict(lds_bvh=0, lds_objects=0)), ((121, 77), 6, 12, dict(leaf=5)),
    ((121, 77), 6, 255, dict(leaf=8, lds_bvh=0)), ((121, 77), 9, 12, dict(pipes=3, queue=4096))])
def test_path_kernel_matches_oracle(size, spp, bounces, opts):
    sc = scenegen.plain_1080p(3, *size)
    print(f"frame {size} spp={spp} bounces={bounces} opts={opts}", flush=True)
    with ra.HipRenderer(max_sample_count=spp, max_bounces=bounces, seed=17, **opts) as r:
        img = r.render_frame(sc)
        acc = r.accumulator()
    ref = oracle.render(sc, spp, bounces, 17)
    np.testing.assert_array_equal(acc.view(np.uint32), ref.view(np.uint32))
    np.testing.assert_array_equal(img.reshape(-1), oracle.tonemap(ref, spp))


@pytest.mark.parametrize("semantics", [0, 1])
@pytest.mark.parametrize("objects,opts", [
    (130, dict()), (185, dict()), (240, dict()), (320, dict()), (2850, dict()), (3200, dict()),
    (185, dict(lds_bvh=14335)), (185, dict(lds_bvh=14336, lds_objects=0)),
    (60, dict(lds_bvh=14335, pipes=3, queue=4096))])
def test_trees_around_what_fits_in_lds(objects, opts, semantics):
    # tree and objects in LDS, the tree alone, neither, by size and by option
    sc = scenegen.clustered(6, objects, 90, 61)
    with ra.HipRenderer(max_sample_count=3, max_bounces=12, seed=3, semantics=semantics, **opts) as r:
        r.render_frame(sc)
        acc = r.accumulator()
    ref = (oracle.render(sc, 3, 12, 3) if semantics == 0 else
           oracle.vk_render(sc, ra.camera_vulkan_inverse_view(sc.camera), 3, 12, threads=8))
    np.testing.assert_array_equal(acc.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("scale,shift", [(1.0, 0.0), (2.0 ** -40, 0.0), (2.0 ** 12, 0.0),
                                         (1.0, 4096.0), (2.0 ** -12, 1.0), (2.0 ** 40, 0.0)])
@pytest.mark.parametrize("objects", [2, 97, 2400, 3200])
def test_compact_tree_at_every_scale(objects, scale, shift):
    # planes are FP16 offsets in a power of two of each node's own from an
    # origin of its own: tiny and huge scenes, scenes far from zero, and the
    # tree's form changing in mid-frame
    sc = scenegen.clustered(6, objects, 70, 41)
    sc.objects["center"] = sc.objects["center"] * np.float32(scale) + np.float32(shift)
    sc.objects["size"] *= np.float32(scale)
    c = sc.camera
    at = [[float(np.float32(v * scale + shift)) for v in c[k]] for k in ("position", "target")]
    sc.camera = scene.make_camera(at[0], at[1], (0, 1, 0), 70, 41, fov_deg=60, near=0.1 * scale, far=100 * scale)
    ref = oracle.render(sc, 4, 12, 3)
    with ra.HipRenderer(max_sample_count=4, max_bounces=12, seed=3, lds_bvh=0) as r:
        r.new_frame(sc)
        for lds in (0, 14336, 0, 14336):
            r.set_option("lds_bvh", lds)
            r.render_sample(sc)
        np.testing.assert_array_equal(r.accumulator().view(np.uint32), ref.view(np.uint32))
        r.new_frame(sc)
        for lds in (14336, 0, 0, 0):
            r.set_option("lds_bvh", lds)
            r.render_sample(sc)
        np.testing.assert_array_equal(r.accumulator().view(np.uint32), ref.view(np.uint32))


def _arithmetic_scene(view, scale):
    # spheres and cubes on and around the camera's axis, with faces in the
    # planes of the camera's position and shared by neighbours
    sc = scenegen.plain_1080p(3, 61, 41)
    sc.objects = np.concatenate([sc.objects, np.array([
        scene.make_object(k, c, size, roughness=0.3, metallic=m)
        for k, c, size, m in [(abi.RD_CUBE, (0, 0.5, 3), 1, 0.0), (abi.RD_CUBE, (1, 0.5, 3), 1, 1.0),
                              (abi.RD_CUBE, (-1, 1.5, 3), 1, 0.0), (abi.RD_SPHERE, (0, 1, 6), 1, 1.0),
                              (abi.RD_SPHERE, (0, 1, 1), 2.0 ** -13, 0.0)]], abi.OBJECT_DTYPE)])
    for f in ("center", "size"):
        sc.objects[f] *= np.float32(scale)
    kw = dict(fov_deg=60) if view == "axis" else dict(ortho_size=6 * scale)
    sc.camera = scene.make_camera((0, scale, -8 * scale), (0, scale, 0), (0, 1, 0), 61, 41,
                                  near=0.1 * scale, far=100 * scale, **kw)
    return sc


@pytest.mark.parametrize("lds_bvh", [0, 1 << 16])
@pytest.mark.parametrize("scale", [2.0 ** -40, 2.0 ** -12, 1.0, 2.0 ** 9, 2.0 ** 30])
@pytest.mark.parametrize("view", ["axis", "parallel"])
def test_walk_arithmetic_at_its_limits(view, scale, lds_bvh):
    # the walk's divisions and roots are exact forms for a range of their
    # arguments and the plain ones outside: zero direction components and
    # numerators, tiny and huge discriminants, rays that no walk takes; trees
    # in memory have the pool of primitives
    sc = _arithmetic_scene(view, scale)
    print(f"arithmetic {view} scale={scale} lds={lds_bvh}", flush=True)
    for semantics in (0, 1):
        with ra.HipRenderer(max_sample_count=3, max_bounces=12, seed=9, semantics=semantics,
                            lds_bvh=lds_bvh) as r:
            r.render_frame(sc)
            acc = r.accumulator()
        ref = (oracle.render(sc, 3, 12, 9) if semantics == 0 else
               oracle.vk_render(sc, ra.camera_vulkan_inverse_view(sc.camera), 3, 12, threads=8))
        np.testing.assert_array_equal(acc.view(np.uint32), ref.view(np.uint32))


def test_path_kernel_and_wavefront_alternate_on_one_renderer():
    # the camera-hit tables of the two are separate: a pass of either must not
    # leave the other with the hits of an earlier frame or scene
    a, b = scenegen.plain_1080p(3, 96, 54), scenegen.clustered(4, 300, 96, 54)
    with ra.HipRenderer(max_sample_count=4, max_bounces=12, seed=5) as r:
        for sc in (a, b):
            r.new_frame(sc)
            for block in (256, 128, 256, 128):  # the path kernel has one workgroup size
                r.set_option("block", block)
                r.render_sample(sc)
            ref = oracle.render(sc, 4, 12, 5)
            np.testing.assert_array_equal(r.accumulator().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("opts", [dict(pipes=1), dict(pipes=1, ticket_cap=3), dict(pipes=2),
                                  dict(pipes=1, queue=4096), dict(pipes=1, l_capacity=1 << 16)])
def test_batch_mixes_path_kernel_and_wavefront_jobs(opts):
    # one streamer's ticket list holds passes of both: a scene without a tree
    # is the wavefront's, the others are the path kernel's
    from raydar_amd.batch import BatchRenderer, Job
    empty = scenegen.plain_small(0)
    empty.objects = empty.objects[:0]
    specs = [(scenegen.clustered(5, 300, 96, 64), 5, 12, 12), (empty, 3, 12, 1),
             (scenegen.plain_1080p(1, 120, 68), 4, 12, 13), (empty, 2, 4, 2),
             (scenegen.plain_1080p(1, 7, 5), 9, 3, 14)]
    jobs = [Job(s, spp, b, seed, pass_samples=2, progress=k % 2 == 0)
            for k, (s, spp, b, seed) in enumerate(specs)]
    with BatchRenderer(**opts) as br:
        for _ in range(2):
            br.render(jobs)
            for job, (s, spp, b, seed) in zip(jobs, specs):
                ref = oracle.render(s, spp, b, seed)
                np.testing.assert_array_equal(job.acc.view(np.uint32), ref.view(np.uint32))
                np.testing.assert_array_equal(job.rgba.reshape(-1), oracle.tonemap(ref, spp))
                job.acc[:] = 0


@pytest.mark.parametrize("size,spp", [((5, 3), 3), ((640, 360), 37), ((2048, 1620), 2),
                                      ((2048, 1650), 2)])
def test_allocation_free_call_matches_render_frame(size, spp):
    # the camera-hit table takes the queues' place in the static scratch while
    # it and a sample of every pixel fit there (images up to 3.3 M pixels: the
    # third size does, the fourth does not), in one pass or several
    sc = scenegen.plain_1080p(3, *size)
    out = np.zeros((sc.height, sc.width, 4), np.uint8)
    f = ra.lib().rd_render_frame_noalloc
    f.restype, f.argtypes = C.c_int, [C.c_void_p, C.POINTER(abi.RdScene), C.c_void_p, C.c_size_t]
    with ra.HipRenderer(max_sample_count=spp, max_bounces=12, seed=5) as r:
        s = sc.as_rd()
        for _ in range(2):
            ra.check(f(r._h, C.byref(s), out.ctypes.data_as(C.c_void_p), out.nbytes), r._h)
        np.testing.assert_array_equal(out, r.render_frame(sc))


@pytest.mark.parametrize("size,spp,bounces,opts", [
    ((1, 1), 9, 12, dict()), ((7, 9), 5, 12, dict()), ((65, 1), 3, 1, dict()),
    ((121, 77), 6, 12, dict(grid=1)), ((121, 77), 6, 12, dict(refill=1)),
    ((121, 77), 6, 12, dict(refill=64, leaf=5)), ((121, 77), 6, 40, dict(lds_bvh=0, lds_objects=0))])
def test_path_kernel_vulkan_semantics_match_oracle(size, spp, bounces, opts):
    # a lane takes its pixel's samples one after another on the pixel's one
    # stream of random numbers
    sc = scenegen.plain_1080p(3, *size)
    print(f"vulkan frame {size} spp={spp} bounces={bounces} opts={opts}", flush=True)
    with ra.HipRenderer(max_sample_count=spp, max_bounces=bounces, semantics=1, **opts) as r:
        img = r.render_frame(sc)
        acc = r.accumulator()
    ref = oracle.vk_render(sc, ra.camera_vulkan_inverse_view(sc.camera), spp, bounces, threads=8)
    np.testing.assert_array_equal(acc.view(np.uint32), ref.view(np.uint32))
    np.testing.assert_array_equal(img.reshape(-1), oracle.vk_tonemap(ref, spp))


@pytest.mark.parametrize("objects", range(1, 10))
def test_nodes_with_each_number_of_leaves(objects):
    # a root of one to four leaves with empty slots, then leaves beside inner
    # children, spheres and cubes in one wave, entered in every combination
    sc = scenegen.plain_1080p(4, 77, 50)
    sc.objects = sc.objects[[0, 65, 1, 66, 2, 67, 3, 68, 4][:objects]]
    with ra.HipRenderer(max_sample_count=4, max_bounces=12, seed=3) as r:
        r.render_frame(sc)
        acc = r.accumulator()
    ref = oracle.render(sc, 4, 12, 3)
    np.testing.assert_array_equal(acc.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("height,scale,shift", [
    (960, 1.0, 0.0), (640, 1.0, 0.0),  # on both sides of where half-size nodes are used
    (960, 2.0 ** -40, 0.0), (960, 2.0 ** 12, 0.0), (960, 1.0, 4096.0), (960, 2.0 ** -12, 1.0), (960, 2.0 ** 40, 0.0)])
def test_large_tree_and_long_pass_at_every_scale(height, scale, shift):
    sc = scenegen.clustered(6, 14000, 1536, height)
    sc.objects["center"] = sc.objects["center"] * np.float32(scale) + np.float32(shift)
    sc.objects["size"] *= np.float32(scale)
    c = sc.camera
    at = [[float(np.float32(v * scale + shift)) for v in c[k]] for k in ("position", "target")]
    sc.camera = scene.make_camera(at[0], at[1], (0, 1, 0), 1536, height, fov_deg=60, near=0.1 * scale,
                                  far=100 * scale)
    with ra.HipRenderer(max_sample_count=2, max_bounces=4, seed=3) as r:
        r.render_frame(sc)
        acc = r.accumulator()
    pix = np.arange(0, 1536 * height, 1999, dtype=np.uint32)
    ref = oracle.render(sc, 2, 4, 3, pixels=pix, threads=8)
    np.testing.assert_array_equal(acc[pix].view(np.uint32), ref.view(np.uint32))
