"""Which form of the skinny GEMM a weight takes (csrc/skinny_form.h), compiled for the host: the shapes
where one form was measured against another take the faster one, and every choice is one the kernels can
run (whole batches or chunks of k per slice). And where the engine takes the kernel rather than hipBLASLt."""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

from kvserve_amd.engine.ops import skinny_wins

CSRC = Path(__file__).resolve().parent.parent / "kvserve_amd/csrc"
FULL, HALF, SHARED = 0, 1, 2

SOURCE = """
#include "skinny_form.h"
extern "C" {
int form(long rows, long k, int m) { return kvh::skinny_form(rows, k, m); }
int slices(long rows, long k, int m) { return kvh::skinny_slices(rows, k, m); }
int batch(int f) { return kvh::skinny_batch((kvh::SkinnyForm)f); }
int chunk() { return kvh::kSkinnyChunk; }
int waves() { return kvh::kSkinnyWaves; }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("form")
    (d / "form.cpp").write_text(SOURCE)
    out = d / "form.so"
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "form.cpp"), "-o", str(out)],
                   check=True)  # fmt: skip
    lib = ctypes.CDLL(str(out))
    lib.form.argtypes = lib.slices.argtypes = [ctypes.c_long, ctypes.c_long, ctypes.c_int]
    return lib


# (rows, k), rows of x, the faster form by 3% or more
MEASURED = [
    ((2048, 2048), 8, HALF), ((1024, 4096), 8, HALF), ((2048, 8192), 5, HALF), ((512, 3072), 8, FULL),
    ((3072, 2048), 8, FULL), ((3072, 4096), 8, FULL), ((4096, 4096), 8, FULL), ((2048, 1024), 8, FULL),
    ((5120, 2048), 5, SHARED), ((6144, 2048), 8, SHARED), ((6144, 4096), 8, SHARED), ((6144, 1024), 8, FULL),
    ((8192, 1024), 5, FULL), ((8192, 1024), 16, FULL), ((8192, 1024), 64, FULL), ((10240, 1024), 24, SHARED),
    ((12288, 1024), 5, FULL), ((12288, 1024), 12, FULL), ((14336, 1024), 16, SHARED), ((16384, 1024), 5, FULL),
    ((16384, 1024), 16, SHARED), ((28672, 1024), 8, SHARED),
    ((8192, 4096), 16, SHARED), ((8192, 2048), 33, FULL), ((8192, 4096), 48, FULL), ((8192, 4096), 64, SHARED),
    ((9216, 2048), 33, SHARED), ((16384, 2048), 64, SHARED), ((128256, 4096), 32, SHARED),
]  # fmt: skip


@pytest.mark.parametrize(("shape", "m", "form"), MEASURED)
def test_measured_shapes_take_the_faster_form(lib, shape, m, form):
    assert lib.form(*shape, m) == form


def test_extra_rounds_are_not_bought(lib):
    assert lib.slices(8192, 4096, 16) == 2 and lib.slices(10240, 1024, 24) == 1 and lib.slices(8208, 4096, 33) == 1


def test_every_choice_can_run(lib):
    for rows in range(16, 20000, 16):
        for k in (1024, 2048, 3072, 4096, 5120, 14336):
            for m in (1, 5, 8, 9, 16, 17, 32, 33, 48, 49, 64):
                f, ks = lib.form(rows, k, m), lib.slices(rows, k, m)
                assert ks == lib.waves() if f != SHARED else ks in ((1, 2) if m <= 32 else (1,))
                assert k % (ks * (lib.chunk() if f == SHARED else lib.batch(f))) == 0
                assert m <= 8 or f != HALF


# rows of x, (n, k), whether the skinny kernel was faster than hipBLASLt (by 3% or more either way)
ROUTED = [
    (8, (4096, 5120), True), (8, (6144, 4096), True), (5, (7168, 4096), True), (8, (2048, 14336), True),
    (8, (7168, 5120), True), (8, (28672, 4096), True), (8, (3584, 11264), False), (16, (4096, 4096), True),
    (16, (3072, 4096), True), (16, (7168, 2048), True), (16, (5120, 3072), False), (16, (6144, 3072), False),
    (16, (5120, 4096), False), (16, (2048, 8192), False), (16, (28672, 4096), True), (32, (3072, 2048), True),
    (32, (4096, 8192), False), (33, (3072, 2048), False),
]  # fmt: skip


@pytest.mark.parametrize(("m", "shape", "wins"), ROUTED)
def test_the_engine_takes_the_faster_kernel(m, shape, wins):
    assert skinny_wins(m, *shape) == wins
