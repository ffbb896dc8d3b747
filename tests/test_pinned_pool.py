"""The pinned pool (csrc/pinned_pool.h) against a host stand-in of the HIP calls it makes: taking
a chunk never asks an event whose stream is being captured or has gone, and no chunk is
handed on while copies read it."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(HERE, "host")


def test_pinned_pool(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text('#include "hip_stand_in.h"\n')
    exe = tmp_path / "pinned_pool"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", str(tmp_path), "-I", HOST,
                    "-I", os.path.join(HERE, "..", "nexus_amd", "csrc"), os.path.join(HOST, "pinned_pool.cpp"), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
