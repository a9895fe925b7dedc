"""The output calls' working memory (csrc/scratch.hip): its bookkeeping, built for the host
against a stand-in for the HIP runtime (tests/c/hip_host), so that the order of waits,
frees and hand-overs can be seen without a GPU."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("scratch") / "scratch_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", os.path.join(HERE, "c", "hip_host"), "-x", "c++",
                    os.path.join(HERE, "c", "scratch_test.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("name", ["waits_for_the_stream", "large_block_leaves_the_others", "oldest_go_first",
                                  "frees_hold_no_lock", "allocation_waits_for_frees", "copy_without_threads",
                                  "kept_memory_is_available", "copies_of_every_length"])
def test_scratch(program, name):
    r = subprocess.run([program, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
