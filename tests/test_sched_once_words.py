"""The words in which the tiles of a striping batch in one launch agree on the scheduler's counters (csrc/sched_once.hpp), in
every order of their steps (tests/host/once_driver.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_counters_are_moved_on_once_whoever_comes_last(tmp_path):
    """The last tile may be done before tile 0 has begun: the counters are moved on all the same, and no tile starts from the
    ones that have been."""
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    exe = os.path.join(tmp_path, "once")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "aws_ofi_nccl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "once_driver.cpp"), "-o", exe], check=True)
    proc = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert proc.returncode == 0 and proc.stdout.endswith("ok\n"), proc.stdout[-4000:]
