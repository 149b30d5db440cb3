"""A batch whose new tile cannot be allocated keeps the tile it had, tables and all
(otherwise a later run would update part of each grid).  CPU only: the driver's own
definitions of the HIP calls stand before the runtime's."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
PKG = ROOT / "euler2d_kokkos_amd"


def test_refused_tile_changes_nothing(tmp_path):
    gxx = shutil.which("g++")
    if not gxx or not (PKG / "libeuler2d_hip.so").exists():
        pytest.skip("g++ or the built library not available")
    exe = tmp_path / "batch_refused_driver"
    res = subprocess.run([gxx, "-std=c++17", "-O1", "-rdynamic", f"-I{ROOT / 'include'}",
                          str(ROOT / "tests" / "host" / "batch_refused_driver.cpp"),
                          f"-L{PKG}", "-leuler2d_hip", f"-Wl,-rpath,{PKG}",
                          "-Wl,--allow-shlib-undefined", "-o", str(exe)],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    deck = tmp_path / "implode.ini"
    deck.write_text("[run]\ntEnd=1.0\nnStepmax=1000\n[mesh]\nnx=128\nny=128\n"
                    "[hydro]\nproblem=implode\n")
    res = subprocess.run([str(exe), str(deck)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, (res.returncode, res.stdout, res.stderr)
    assert "refused tiles change nothing" in res.stdout
