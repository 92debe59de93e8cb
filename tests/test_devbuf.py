"""The workspaces' growth (csrc/devbuf.hip) on a device with little room,
compiled for the host over fake HIP calls."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_workspace_growth_keeps_what_it_has(tmp_path):
    exe = str(tmp_path / "devbuf_test")
    csrc = os.path.join(ROOT, "go-infer_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                    "-I" + os.path.join(HERE, "c", "fakehip"), "-I" + csrc, "-I" + os.path.join(ROOT, "include"),
                    "-x", "c++", os.path.join(csrc, "devbuf.hip"), os.path.join(HERE, "c", "devbuf_test.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
