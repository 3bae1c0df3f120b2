"""The rule that admits launches whose blocks wait for each other (host)."""
import ctypes
import os
import subprocess

from damascene_amd._lib import lib

HERE = os.path.dirname(os.path.abspath(__file__))


def test_gate_rules(tmp_path):
    exe = str(tmp_path / "resident_gate_check")
    subprocess.run(["g++", "-std=c++17", "-O1", os.path.join(HERE, "resident_gate_check.cpp"), "-o", exe,
                    "-lpthread"], check=True)
    assert subprocess.run([exe]).returncode == 0


def test_report_rejects_bad_arguments():
    v = ctypes.c_int()
    assert lib().dmsc_resident_report(None, ctypes.byref(v), ctypes.byref(v)) == 1
