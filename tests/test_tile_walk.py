"""The index arithmetic of the persistent matmul kernels (catccos_amd/csrc/tile_walk.h), walked on the host: every tile goes to one
workgroup, whatever the number of CUs, and every slab that they ask memory for lies within K, whatever the number of slabs."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_walk_stays_in_range(tmp_path):
    exe = str(tmp_path / "walk_model")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", os.path.join(HERE, "csrc", "walk_model.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-3000:]
