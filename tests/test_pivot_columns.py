"""The barriers of the small-front column loop (csrc/mf_pivots.h), run on the host in many orders
of its four wavefronts: a failed pivot ends the front for all of them at the same barrier."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "cliquetrees.jl_amd", "csrc")


def test_failed_pivot_ends_every_wavefront_together(tmp_path):
    exe = str(tmp_path / "pivot_columns")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "pivot_columns.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
