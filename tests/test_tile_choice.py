"""CPU test of the shortened choice of the pair form's tiles
(tests/cpp/tile_choice_check.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest


def test_tile_choice(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    repo = Path(__file__).resolve().parent.parent
    csrc = repo / "cice-evp1d_amd" / "csrc"
    exe = tmp_path / "choice"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", f"-I{csrc}",
                    str(repo / "tests" / "cpp" / "tile_choice_check.cpp"), str(csrc / "evp1d_tiles.cpp"), "-o",
                    str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
