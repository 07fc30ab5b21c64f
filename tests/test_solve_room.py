"""The workspaces of a solve (csrc/mf_room.h) against memories that are too small, on the host."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "cliquetrees.jl_amd", "csrc")


def test_workspaces_of_a_solve(tmp_path):
    exe = str(tmp_path / "solve_room")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "solve_room.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
