"""The block cache behind device allocations, on the CPU:
tests/block_cache_host.cpp runs it over a memory that counts allocations,
frees and synchronisations."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("block_cache") / "block_cache_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-Wall",
                    "-I", os.path.join(HERE, "..", "qopqdp_amd", "csrc"),
                    os.path.join(HERE, "block_cache_host.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("check", ["freed_blocks_wait_for_a_sync", "nobody_waits_behind_a_sync",
                                   "nobody_waits_behind_a_free", "blocks_have_one_owner",
                                   "blocks_are_little_larger_than_asked", "kept_memory_is_bounded",
                                   "failed_allocations_give_kept_blocks_back"])
def test_block_cache(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
