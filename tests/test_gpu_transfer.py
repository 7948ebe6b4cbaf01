"""Host copies through an engine's pinned buffers (transfer.hpp): images and
accumulators whose bytes end at, before and behind the edges of a part, a slot
and the ring, and scenes below and above what an upload gathers."""
import numpy as np
import pytest

import oracle
import raydar_amd as ra
from raydar_amd import scenegen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height", [
    (1, 1), (127, 129), (128, 128), (128, 129),  # 256 KiB of accumulator
    (255, 257), (256, 256), (256, 257),          # 1 MiB of it: threads; 256 KiB of image
    (512, 257), (512, 512), (513, 512),          # 2 and 4 MiB: slots; 1 MiB of image
    (1024, 512), (1024, 513), (1031, 1030)])     # 8 MiB: the ring once, and round again
def test_reads_around_the_edges_of_parts_slots_and_ring(width, height):
    sc = scenegen.plain_1080p(1, width, height)
    with ra.HipRenderer(max_sample_count=2, max_bounces=2, seed=3) as r:
        for seed in (3, 4):
            r.set_seed(seed)
            img = r.render_frame(sc)
            acc = r.accumulator()
            ref = oracle.render(sc, 2, 2, seed)
            np.testing.assert_array_equal(acc.view(np.uint32), ref.view(np.uint32))
            np.testing.assert_array_equal(img.reshape(-1), oracle.tonemap(ref, 2))


def test_scenes_of_growing_size_through_one_renderer():
    with ra.HipRenderer(max_sample_count=1, max_bounces=4, seed=3) as r:
        for n in [0, 1, 300, 1000, 1000, 1000, 14000, 20000, 5]:  # to 4 MB and above
            sc = scenegen.clustered(2, max(n, 1), 40, 30)
            sc.objects = sc.objects[:n]
            r.render_frame(sc)
            ref = oracle.render(sc, 1, 4, 3)
            np.testing.assert_array_equal(r.accumulator().view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("semantics", [0, 1])
@pytest.mark.parametrize("width,height,per_pass", [
    (1, 1, 2), (511, 512, 2), (512, 512, 1), (513, 512, 2)])  # images written by the device below 1 MiB
def test_image_of_every_pass_around_the_direct_limit(width, height, per_pass, semantics):
    sc = scenegen.plain_1080p(1, width, height)
    spp = 4
    with ra.HipRenderer(max_sample_count=spp, max_bounces=3, seed=5, semantics=semantics,
                        l_capacity=max(1 << 16, width * height)) as r:  # a pass holds one sample
        r.set_samples_per_pass(per_pass)
        r.new_frame(sc)
        step = spp if semantics else per_pass
        for done in range(step, spp + 1, step):
            img = r.render_sample()
            if semantics:
                ref = oracle.vk_render(sc, ra.camera_vulkan_inverse_view(sc.camera), done, 3, threads=8)
                want = oracle.vk_tonemap(ref, done)
            else:
                ref = oracle.render(sc, done, 3, 5, threads=8)
                want = oracle.tonemap(ref, done)
            np.testing.assert_array_equal(r.accumulator().view(np.uint32), ref.view(np.uint32))
            np.testing.assert_array_equal(img.reshape(-1), want)
            assert r.sample_count == done
