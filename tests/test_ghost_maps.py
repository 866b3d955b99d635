"""The ghosts that the fused stages write along with the active cells are those
of the ghost fill: the kernels' own maps, compiled for the host, over every
boundary and the smallest sizes (tests/ghost_maps.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_scattered_ghosts_are_the_fills(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "ghost_maps")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17",
                    os.path.join(HERE, "ghost_maps.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert r.stdout.endswith("grids, 0 differences\n")
