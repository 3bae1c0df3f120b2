"""The walk rules compiled into the affinity kernel, over every window (host)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_walk_rules_cover_every_window(tmp_path):
    exe = str(tmp_path / "walks_check")
    subprocess.run(["g++", "-std=c++17", "-O1", os.path.join(HERE, "walks_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "1296 windows\n", r.stdout
