"""The library's allocation and error paths on the CPU: test programs define the HIP calls themselves (tests/host)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def _run(sg, tmp_path, name):
    exe = tmp_path / name
    libdir = os.path.dirname(sg.LIB_PATH)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-rdynamic", "-I", os.path.join(ROOT, "include"), "-I",
                    "/opt/rocm/include", os.path.join(HERE, "host", name + ".cpp"), "-L", libdir, "-lsgtsne_hip",
                    "-Wl,-rpath," + libdir, "-Wl,--allow-shlib-undefined", "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("name", ["lost_blocks", "block_cache_oom", "sticky_error", "exact_rows_memory", "block_cache_bounds", "pool_kept"])
def test_host_program(sg, tmp_path, name):
    _run(sg, tmp_path, name)
