"""Which workgroups of a launch take part in a panel on one die (csrc/elect.hpp): all the
places of one die, each once, whoever starts late and whatever has been reported by then;
and each workgroup decides once, in one thread."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_places_under_random_starts_and_a_failure(tmp_path):
    exe = tmp_path / "elect_model"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I",
                    os.path.join(ROOT, "scirs_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "elect_model.cpp"),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.startswith("ok"), out.stdout


def test_no_wave_of_a_many_workgroup_panel_decides_by_itself():
    """The panel reports a failure while workgroups of the same launch still start: ahead of
    the election (and outside the one-workgroup form) no wave may look at the flag."""
    with open(os.path.join(ROOT, "scirs_amd", "csrc", "subpanel.hip")) as f:
        src = f.read()
    body = src[src.index("void sub_panel_kernel("):]
    head = body[:body.index("} else {")]
    assert "elect::place" in head and not re.search(r"\*\s*A\.info", head)
