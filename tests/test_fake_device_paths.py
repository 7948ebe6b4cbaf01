"""The library's host code on the fake HIP device with the path kernel among the
fake kernels (tests/fakehip/fake_paths.cpp): the route nearly every scene takes
on a GPU (run_paths, its camera-hit tables, half-size trees and work lists, the
streams it is spread over, the batch's passes launched as they are issued, the
image queued with its pass), under AddressSanitizer + UndefinedBehaviorSanitizer
and ThreadSanitizer.  test_fake_device.py runs the wavefront throughout."""
import pytest

from tests.test_fake_device import _build, _run


@pytest.fixture(scope="module")
def asan(tmp_path_factory):
    return _build(str(tmp_path_factory.mktemp("fakepaths")), "paths_asan")


@pytest.fixture(scope="module")
def tsan(tmp_path_factory):
    return _build(str(tmp_path_factory.mktemp("fakepaths_tsan")), "paths_tsan")


@pytest.mark.parametrize("args,nosync", [(["path_frames"], "1"), (["plain"], "0"), (["noalloc"], "1"),
                                         (["batch"], "1"), (["path_budget"], "1"),
                                         (["noalloc_large"], "0"), (["lds_limit"], "0"), (["no_memory"], "0"),
                                         (["no_image"], "0"), (["new_scenes"], "1"),
                                         (["server", "--seconds", "20", "--speed", "20"], "1")])
def test_path_kernel_host_code_asan(asan, args, nosync):
    _run(asan, args, 900, FAKEHIP_FREE_NOSYNC=nosync)


@pytest.mark.parametrize("args", [["path_frames"], ["plain"]])
def test_path_kernel_host_code_tsan(tsan, args):
    _run(tsan, args, 900)


def test_autotune_results_of_the_wavefront_alone_are_not_taken(asan, tmp_path):
    # a file of results from before the path kernel (lines whose key does not
    # name the kernels): a workgroup size that was best then would keep a batch
    # off the path kernel
    f = tmp_path / "tune.txt"
    _run(asan, ["autotune"], 900, RAYDAR_HIP_TUNE_CACHE=str(f))
    lines = f.read_text().splitlines()
    old = [l.replace("|kernels=paths", "") for l in lines]
    f.write_text("\n".join(old) + "\n")
    again = _run(asan, ["autotune"], 900, RAYDAR_HIP_TUNE_CACHE=str(f))
    assert "autotune cached=0" in again and "other mix cached=0" in again
    assert f.read_text().splitlines()[:2] == old
