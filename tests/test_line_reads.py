"""Where the decode kernels read K in whole lines (csrc/line_reads.h), compiled for the host: measured shapes
take the faster reads, and the stream-K decode's choice is one for the whole launch."""

from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "kvserve_amd/csrc"

SOURCE = """
#define KVH_LINE_FN static inline
#include "line_reads.h"
extern "C" {
int launch(int D, int rows, long bytes) { return kvh::line_launch(D, rows, bytes); }
int units(int kv8, long C, long n) { return kvh::line_units(kv8, C, n); }
int brief(int D, int kv8, long rows, long tokens) { return kvh::line_short(D, kv8, rows, tokens); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("lines")
    (d / "lines.cpp").write_text(SOURCE)
    out = d / "lines.so"
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "lines.cpp"), "-o", str(out)],
                   check=True)  # fmt: skip
    lib = ctypes.CDLL(str(out))
    lib.launch.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_long]
    lib.units.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_long]
    lib.brief.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_long]
    return lib


# kv heads, head size, bytes an element, most query rows, chunks a unit, whether whole lines were no slower
STREAM = [
    (8, 128, 2, 4, 4, True), (8, 128, 2, 8, 16, True), (4, 128, 2, 4, 8, True), (12, 128, 2, 4, 24, True),
    (8, 128, 2, 4, 73, False), (16, 128, 2, 2, 16, False), (32, 128, 2, 4, 16, False), (1, 128, 2, 8, 12, False),
    (2, 128, 2, 4, 16, False), (8, 64, 2, 4, 3, False), (4, 64, 2, 4, 16, False), (8, 128, 2, 12, 16, False),
    (8, 128, 1, 4, 16, True), (12, 128, 1, 4, 24, True), (16, 128, 1, 2, 12, True), (8, 128, 1, 4, 4, False),
    (4, 128, 1, 4, 24, False), (32, 128, 1, 1, 24, False), (2, 128, 1, 4, 12, False),
]  # fmt: skip


@pytest.mark.parametrize(("kv_heads", "D", "elem", "rows", "unit", "lines"), STREAM)
def test_stream_k_units_take_the_faster_reads(lib, kv_heads, D, elem, rows, unit, lines):
    # the launcher's half of the choice, then the kernel's, over the launch's totals
    chosen = lib.launch(D, rows, kv_heads * D * elem) and lib.units(elem == 1, unit * 128, 128)
    assert bool(chosen) == lines


# sequences, kv heads, head size, E4M3, keys a table holds, whether whole lines were no slower
SHORT = [
    (128, 8, 128, 0, 1008, True), (16, 8, 128, 0, 512, True), (8, 8, 64, 0, 512, False), (32, 8, 128, 1, 1008, False),
    (128, 8, 128, 1, 1008, True), (128, 4, 128, 1, 1008, True), (131, 8, 128, 1, 320, False), (64, 8, 64, 1, 1008, False),
    (96, 8, 128, 1, 1024, True),
]  # fmt: skip


@pytest.mark.parametrize(("B", "kv_heads", "D", "e4m3", "tokens", "lines"), SHORT)
def test_short_decode_takes_the_faster_reads(lib, B, kv_heads, D, e4m3, tokens, lines):
    assert bool(lib.brief(D, e4m3, B * kv_heads * D, tokens)) == lines


def test_the_choice_follows_the_mean_unit(lib):
    # units of 31 and 33 chunks in one launch (64 of each, mean 32) choose together
    assert lib.units(0, 64 * 31 + 64 * 33, 128) and not lib.units(0, 64 * 31 + 64 * 33 + 1, 128)
    assert lib.units(1, 128 * 8 + 1, 128) and not lib.units(1, 128 * 8, 128)
