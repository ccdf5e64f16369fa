"""Where a SIR plan's parts lie in its one buffer (plan_layout.hpp): what the
work-groups read shares no line with what they write by atomics."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_parts_share_no_line(tmp_path):
    exe = str(tmp_path / "plan_layout_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(HERE, "..", "dream_amd", "csrc"),
                    os.path.join(HERE, "cxx", "plan_layout_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["0", "0"]
