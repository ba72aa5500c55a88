"""The drain's derivation of eight descriptors at a time (csrc/gin_derive8.hpp) against the one that takes them one by one,
built with the sanitizers (tests/host/derive8_driver.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "aws_ofi_nccl_amd", "csrc")


def test_eight_descriptors_at_a_time_are_derived_as_one_by_one(tmp_path):
    """Sizes around every threshold and up to 2^64 - 1, all rail counts of the fast form, pins and runs that come in and
    reach their end, regions alike and mixed, signals, the window near its limit, descriptors that are handed back; groups that
    a ring's end or 2^32 cuts, arrays of records at any 8-byte offset, drains that end at a bad descriptor."""
    if not shutil.which("g++"):
        pytest.skip("no host compiler")
    exe = os.path.join(tmp_path, "derive8")
    subprocess.run(["g++", "-std=c++17", "-pthread", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-static-libasan", "-static-libubsan", "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(ROOT, "tests", "host", "derive8_driver.cpp"),
                    *[os.path.join(CSRC, s) for s in ("gin_proxy.cpp", "gin_wire.cpp", "sched_host.cpp")], "-o", exe], check=True)
    proc = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    if "skip" in proc.stdout:
        pytest.skip("no AVX-512 here")
    assert proc.returncode == 0 and "ok: " in proc.stdout, proc.stdout[-4000:]
