"""HostLink's control flow on the CPU (tests/xfer_host.cpp on tests/fake_hip):
with pinned memory, with none, and with only a little; late streams; host arrays
reused right after an upload; threads."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_transfers_on_a_late_stream(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no g++")
    exe = str(tmp_path / "xfer_host")
    subprocess.run([cxx, "-std=c++17", "-O1", "-g", "-pthread", "-fsanitize=address,undefined",
                    "-I", os.path.join(HERE, "fake_hip"), os.path.join(HERE, "xfer_host.cpp"),
                    "-o", exe], check=True)
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")  # a preloaded library is fine
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout == "0 failures\n"
