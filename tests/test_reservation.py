"""The reservation of a device's waves under contention (host code)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_requests_do_not_refuse_each_other(tmp_path):
    exe = str(tmp_path / "reservation")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-pthread",
                    "-I" + os.path.join(ROOT, "eikonalxx_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "reservation.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
