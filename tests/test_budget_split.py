"""The budget's split of a layer over threads: every node once, workgroups full whatever the
row length, and no chain of rows where the launch does not fill the GPU (built for the host
against tests/c/hip_host)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_budget_split(tmp_path):
    exe = str(tmp_path / "budget_split_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(HERE, "c", "hip_host"),
                    os.path.join(HERE, "c", "budget_split_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
