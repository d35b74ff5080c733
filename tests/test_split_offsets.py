"""The source offsets of the general limb split (csrc/tamx_offsets.hpp) on
the host, built with g++ -fsanitize=undefined: a tile without rows or k has
modes of extent zero, which must not be divided by."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_offsets_of_empty_and_ragged_tiles(tmp_path):
    exe = tmp_path / "split_offsets"
    r = subprocess.run(["g++", "-std=c++17", "-w", "-g", "-O1", "-D__HIP_PLATFORM_AMD__",
                        "-fsanitize=undefined", "-fno-sanitize-recover=all",
                        "-I", "/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "tiledarray_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "split_offsets.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.stdout + r.stderr)[-3000:]
    assert "OFFSETS OK" in r.stdout
