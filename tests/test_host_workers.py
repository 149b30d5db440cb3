"""The helper threads of the host copies: when the memory for a thread's start is
refused, its share runs on the caller's thread and the process goes on (an
exception past running threads would end it).  CPU only; needs g++."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_refused_thread_starts(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = tmp_path / "workers_driver"
    res = subprocess.run([gxx, "-std=c++17", "-O1", "-pthread",
                          f"-I{ROOT / 'euler2d_kokkos_amd' / 'csrc'}",
                          str(ROOT / "tests" / "host" / "workers_driver.cpp"), "-o", str(exe)],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, (res.returncode, res.stdout, res.stderr)
    assert "every share ran once" in res.stdout
