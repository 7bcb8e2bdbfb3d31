"""The tags of the words that a panel's waves exchange (csrc/tags.hpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_earlier_word_passes_for_a_current_one(tmp_path):
    exe = tmp_path / "tags_model"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "scirs_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "tags_model.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout
