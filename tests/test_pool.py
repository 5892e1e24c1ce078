"""Kept device blocks on the CPU: device_pool.cpp with an allocator of the test
in place of the device's (tests/cpp/pool_main.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def pool_exe(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pool") / "pool_main")
    cpp, csrc = os.path.join(ROOT, "tests", "cpp"), os.path.join(ROOT, "naga_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-D__HIPCC__", "-o", exe,
                    os.path.join(cpp, "pool_main.cpp"), os.path.join(csrc, "device_pool.cpp"),
                    "-I", os.path.join(cpp, "fake_hip"), "-I", csrc], check=True)
    return exe


@pytest.mark.parametrize("check", ["eviction", "waiting", "trimming", "exhaustion",
                                   "many_blocks", "threads"])
def test_kept_blocks(pool_exe, check):
    r = subprocess.run([pool_exe, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
