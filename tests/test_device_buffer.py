"""The buffers that captured graphs may hold the address of
(adaptq_amd/csrc/device_buffer.hpp): whatever sizes the calls ask for, an address
once handed out stays allocated until release, and what is kept is bounded
(tests/cpp/device_buffer_check.cpp, over an allocator that keeps books)."""
import os
import shutil
import subprocess

import pytest

from adaptq_amd.build import ROCM

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_addresses_stay(tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    exe = tmp_path / "device_buffer_check"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__",
                        "-I", os.path.join(ROCM, "include"),
                        os.path.join(ROOT, "tests", "cpp", "device_buffer_check.cpp"),
                        "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
