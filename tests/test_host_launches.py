"""What the library launches, without a GPU: the built library runs against a stand-in for the HIP runtime
(tests/host/launch_driver.cpp) that sees every launch's grid and arguments and can refuse a call."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBDIR = os.path.join(ROOT, "aws_ofi_nccl_amd", "lib")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    if not os.path.exists(os.path.join(LIBDIR, "libofi_amd_hotpath.so")):
        from aws_ofi_nccl_amd import build
        build.build_library()
    exe = os.path.join(tmp_path_factory.mktemp("launches"), "launch_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host", "launch_driver.cpp"),
                    "-rdynamic", "-pthread", "-L", LIBDIR, "-l:libofi_amd_hotpath.so", "-Wl,-rpath," + LIBDIR, "-Wl,-rpath,/opt/rocm/lib",
                    "-Wl,--allow-shlib-undefined", "-o", exe], check=True)
    return exe


def run(driver, part):
    proc = subprocess.run([driver, part], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert proc.returncode == 0 and part + ": ok" in proc.stdout, proc.stdout[-4000:]


def test_small_striping_batches_never_meet_a_count_left_by_another(driver):
    """The one-launch form of striping counts its workgroups in a word of the scratch: consecutive batches use
    different words, a count left in one is gone before its turn comes again, and a batch that is captured
    counts in none."""
    run(driver, "striping")


def test_striping_scratch_is_kept_by_stream_and_not_by_handle(driver):
    """hipStreamPerThread and the null stream are one handle for several streams, whose batches may overlap."""
    run(driver, "streams")


def test_copy_tables_of_many_pieces_stay_within_what_a_launch_can_number(driver):
    """A launch holds fewer than 2^32 work-items: tables beyond go in several, up to the documented 2^31 - 1
    pieces, and every entry is in exactly one of them."""
    run(driver, "pieces")


def test_a_bounce_batch_is_launched_alike_whatever_the_size_of_the_pool(driver):
    """The bytes of the source are no measure of the buffers' lengths: short buffers out of a pool are not taken for
    long ones."""
    run(driver, "bounce")


def test_model_grids_that_are_mostly_evaluated_stay_with_small_workgroups(driver):
    """The form for large outputs suits grids that are mostly written."""
    run(driver, "model")


def test_region_tiles_fit_short_axes(driver):
    """A region grid of one size and many node counts, or the other way round, is not paid for by the square."""
    run(driver, "tiles")


def test_an_upload_that_failed_is_made_again(driver):
    """The tuner's grids send a list only when it differs from the last one: one that failed on the way does not
    count as sent."""
    run(driver, "uploads")
