"""A layer's backward pass over interfaces of the caller's own, on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
PKG = os.path.join(ROOT, "sparseconvnet-archived_amd")


def test_interfaces_need_not_be_the_batch_s(tmp_path):
    exe = str(tmp_path / "foreign")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(PKG, "host"), "-I", os.path.join(ROOT, "include"),
                           os.path.join(HERE, "foreign_interface_harness.cpp"), "-o", exe, "-L" + PKG, "-lscn_host", "-lscn_hip",
                           "-Wl,-rpath," + PKG])
    assert subprocess.run([exe], stdout=subprocess.DEVNULL).returncode == 0
