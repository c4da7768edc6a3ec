"""The engine's device memory pool on the host (tests/pool_check.cpp), with a
device of a set size in place of HIP's."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def pool_check(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("g++ or the HIP headers not found")
    exe = str(tmp_path_factory.mktemp("pool") / "pool_check")
    subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-Wall", "-Wno-unused-result", "-pthread",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "pool_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("name", [
    "cached_is_trimmable", "slab_tails_are_used", "block_is_kept", "small_blocks_are_buffers",
    "block_yields_to_its_pool",
    "quarter_stays_free", "block_is_carved", "block_ranges_join",
    "block_and_captures", "block_given_back_in_a_capture",
    "trim_in_a_capture", "block_yields_to_other_pools", "block_from_threads"])
def test_pool(pool_check, name):
    r = subprocess.run([pool_check, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
