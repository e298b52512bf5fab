"""CPU: the tile order of a terrain's cells is a bijection with an inverse, in
square blocks with at most 1/16 unused indices, or x-major (shy_device.hpp:
tile_map, tile_index, tile_xy).  Compiled for the host with g++ from the
header the kernels use."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SIZES = [(1, 1), (1, 500), (500, 1), (3, 9), (4, 8), (5, 8), (64, 64), (65, 64), (64, 100),
         (100, 17), (200, 200), (256, 256), (701, 1103), (1024, 1024), (1000, 700), (37, 2049)]


def test_tile_order_bijection(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    exe = str(tmp_path / "tile_order")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__",
                    "-w", "-o", exe, os.path.join(HERE, "tile_order_check.cpp")], check=True)
    out = subprocess.run([exe] + [str(v) for s in SIZES for v in s], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
