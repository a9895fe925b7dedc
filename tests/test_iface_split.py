"""How the interface fill shares a tile's directions out over workgroups: on every measured
launch within 3% of the fastest number, and no slower than the fill by single directions
was (built for the host)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_iface_split(tmp_path):
    exe = str(tmp_path / "iface_split_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", os.path.join(HERE, "c", "iface_split_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
