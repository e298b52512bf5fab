"""CPU: the walk of one wave per drop addresses every record of the terrains it
takes, and takes no terrain whose records lie beyond 32-bit offsets (odd sides
pad a map of the largest legal size, 2^27 cells, to more than 2^27 records).
Compiled for the host with g++ from the header the kernels use."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
# size, taken
SIZES = [((1, 1), 1), ((2, 300), 1), ((255, 256), 1), ((701, 1103), 1), ((11584, 11584), 1),
         ((11586, 11584), 1),         # 134212224 records
         ((11585, 11585), 0),         # 134212225 cells, 134235396 records
         ((33, 4067100), 0), ((32, 4194304), 1), ((4194304, 32), 1), ((31, 4194303), 1),
         ((4194305, 31), 0), ((1, 134217727), 0)]


def test_solo_record_offsets(tmp_path):
    if shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"):
        pytest.skip("needs g++ and the HIP headers")
    exe = str(tmp_path / "solo_offsets")
    subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-w", "-o", exe, os.path.join(HERE, "solo_offsets_check.cpp")], check=True)
    r = subprocess.run([exe] + [str(v) for s, _ in SIZES for v in s], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert r.stdout.strip() == "".join(str(t) for _, t in SIZES)
