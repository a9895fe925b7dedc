"""Which path a gratio-2 handle takes for its bands: on every measured size within 8% of the
fastest of the three, and no slower than the tiles that served all sizes before (built for
the host)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_band2_pick(tmp_path):
    exe = str(tmp_path / "band2_pick_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", os.path.join(HERE, "c", "band2_pick_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
