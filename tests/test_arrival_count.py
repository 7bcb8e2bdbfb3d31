"""The count by which the workgroups of a launch find out who is the last (csrc/arrive.hpp):
zero again after every launch, also when one of them reports a failure before another starts."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_order_of_start_registration_and_failure(tmp_path):
    exe = tmp_path / "arrive_model"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "scirs_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "arrive_model.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout
