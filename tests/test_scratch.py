"""The device scratch that threads keep between calls (scratch.hpp) against a
small memory on the CPU: idle buffers, of any thread, are given back before an
allocation fails, busy ones and other devices' never; four threads at once."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_scratch_pool(tmp_path):
    exe = str(tmp_path / "scratch_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread",
                    "-I", os.path.join(HERE, "..", "dream_amd", "csrc"),
                    os.path.join(HERE, "cxx", "scratch_check.cc"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True)
    assert out.stdout.split() == ["0"], out.stderr
