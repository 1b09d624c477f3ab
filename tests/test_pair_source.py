"""CPU test of the pair tables' source slots, which launches read in place of
copied ghosts (tests/cpp/pair_source_check.cpp)."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

import evp1d
from evp1d import layout, synth


def test_source_slots(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    repo = Path(__file__).resolve().parent.parent
    csrc = repo / "cice-evp1d_amd" / "csrc"
    exe = tmp_path / "sources"
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", f"-I{csrc}", str(repo / "tests" / "cpp" / "pair_source_check.cpp"),
                    str(csrc / "evp1d_tiles.cpp"), "-o", str(exe)], check=True, capture_output=True)
    g = synth.make_grid(200, 150, 72)
    s = layout.pack(g, evp1d.build_index(g.tmask, g.nghost))
    skip = (s["skipT"] != 0).astype(np.uint8) | ((s["skipU"] != 0).astype(np.uint8) << 1)
    with open(tmp_path / "in.bin", "wb") as fh:
        fh.write(np.array([s["na"], s["navel"]], np.int32).tobytes())
        for n in evp1d.NBR:
            fh.write((s["idx"][n].astype(np.int32) - 1).tobytes())
        fh.write(skip.tobytes())
    r = subprocess.run([str(exe), str(tmp_path / "in.bin")], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
