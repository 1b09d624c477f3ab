"""The library's host side on a HIP runtime without a GPU (tests/cpp/
fake_hip.cpp): its sources compiled for the host only and linked with that
runtime, bound in place of the product's library."""
import ctypes
import re
import shutil
import subprocess
from contextlib import contextmanager
from pathlib import Path

import pytest

import evp1d
from evp1d import build

REPO = Path(__file__).resolve().parent.parent
FLAGS = {False: "libevp1d.so", True: "libevp1d_fma.so"}


class FakeHip:
    """Which kernels calls launched, and allocations made to fail."""

    def __init__(self, lib: ctypes.CDLL):
        self.L = lib
        lib.fake_fail.argtypes = [ctypes.c_long, ctypes.c_long]
        lib.fake_launches.restype = lib.fake_attributes.restype = ctypes.c_char_p
        lib.fake_live.restype = ctypes.c_long

    def fail(self, after: int, count: int = 1) -> None:
        """Of the allocations from now on, `count` fail after the first `after`."""
        self.L.fake_fail(after, count)

    def no_fail(self) -> None:
        self.L.fake_fail(-1, 0)

    def launches(self) -> list:
        """(kernel, workgroups, threads, LDS bytes) since the last call."""
        rows = (r.split("|") for r in self.L.fake_launches(1).decode().splitlines())
        return [(n, int(g), int(b), int(lds)) for n, g, b, lds in rows]

    def kernels(self) -> list:
        return [r[0] for r in self.launches()]

    def attributes(self) -> list:
        """(kernel, LDS bytes) of every hipFuncSetAttribute call."""
        rows = (r.split("|") for r in self.L.fake_attributes().decode().splitlines())
        return [(n, int(v)) for n, v in rows]

    def live(self) -> int:
        return self.L.fake_live()


def build_fake(tmp: Path, fma: bool = False) -> Path:
    if shutil.which(build.HIPCC) is None:
        pytest.skip("hipcc not available")
    csrc = build.CSRC
    objs = []
    for src in [csrc / s for s in build.HIP_SOURCES] + [REPO / "tests" / "cpp" / "fake_hip.cpp"]:
        obj = tmp / (src.stem + ".o")
        subprocess.run([build.HIPCC, "--cuda-host-only", "-O1", "-std=c++17", f"--offload-arch={build.ARCH}", "-fPIC",
                        *build.FLAVOURS[FLAGS[fma]], f"-I{build.INCLUDE}", "-c", str(src), "-o", str(obj)],
                       check=True, capture_output=True)
        objs.append(str(obj))
    und = subprocess.run(["nm", "-u", *objs], check=True, capture_output=True, text=True).stdout
    none = [f"-Wl,--defsym,{s}=0" for s in sorted(set(re.findall(r"__hip_fatbin_\w+", und)))]
    lib = tmp / "libevp1d_fake.so"
    subprocess.run(["g++", "-shared", "-pthread", "-Wl,-Bsymbolic", "-Wl,-z,defs", *none, *objs, "-o", str(lib)],
                   check=True, capture_output=True)
    return lib


@contextmanager
def bound(path: Path, fma: bool = False):
    """The library at `path` in place of the product's for the engines made inside."""
    kept = dict(evp1d._libs)
    try:
        yield FakeHip(evp1d.load(fma, path))
    finally:
        evp1d._libs.clear()
        evp1d._libs.update(kept)


@pytest.fixture(scope="session")
def fake_lib(tmp_path_factory):
    return build_fake(tmp_path_factory.mktemp("fake_hip"))


@pytest.fixture
def fake(fake_lib):
    with bound(fake_lib) as f:
        f.launches()
        yield f
        f.no_fail()
