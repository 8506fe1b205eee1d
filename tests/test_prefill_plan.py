"""The prefill part's flat space of positions (csrc/prefill_plan.h), compiled for the host and
compared with a walk over every tile: the closed form of the tiles' positions, and that it takes a
few steps whatever the prompt's length, for every group size."""

from __future__ import annotations

import ctypes
import random
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "kvserve_amd/csrc"

SOURCE = """
#define KVH_PLAN_FN static inline
#include "prefill_plan.h"
using namespace kvh;
extern "C" {
int tile_cost() { return kTileCost; }
int chunks(int R, int q, int kv, int64_t ctx, int G, int PR, int t) { return pre_tile_chunks({R, q, kv, ctx}, G, PR, t); }
static long entered;  // functions entered since the last count (-finstrument-functions)
__attribute__((no_instrument_function)) void __cyg_profile_func_enter(void*, void*) { ++entered; }
__attribute__((no_instrument_function)) void __cyg_profile_func_exit(void*, void*) {}
__attribute__((no_instrument_function)) long count() { long n = entered; entered = 0; return n; }
int64_t prefix(int R, int q, int kv, int64_t ctx, int G, int PR, int t) { return pre_prefix({R, q, kv, ctx}, G, PR, PR % G == 0 ? PR / G : 0, t); }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    out = d / "plan.so"
    subprocess.run([cxx, "-std=c++17", "-O1", "-finstrument-functions", "-shared", "-fPIC", "-Wl,-Bsymbolic",
                    f"-I{CSRC}", str(d / "plan.cpp"), "-o", str(out)], check=True)  # fmt: skip
    lib = ctypes.CDLL(str(out))
    lib.prefix.restype = ctypes.c_int64
    lib.count.restype = ctypes.c_long
    i, l = ctypes.c_int, ctypes.c_int64
    lib.chunks.argtypes = lib.prefix.argtypes = [i, i, i, l, i, i, i]
    return lib


@pytest.mark.parametrize("PR", [128, 192])
@pytest.mark.parametrize("G", [1, 2, 3, 4, 5, 6, 7, 8, 10, 16, 48, 63, 64])
def test_positions_match_a_walk_over_the_tiles(plan, G, PR):
    rng = random.Random(G * 1000 + PR)
    shapes = [(q, c, q + c) for q in (1, 5, PR // G or 1, PR // G + 1, 2 * PR // G + 1, 700) for c in (0, 1, 31, 32, 4095)]
    shapes += [(rng.randint(1, 1500), rng.randint(0, 20000), None) for _ in range(20)]
    # lengths a broken caller may pass: fewer keys than queries, a block table that ends early
    shapes += [(300, -100, 200), (300, 500, 640), (64, -64, 0)]
    for q, ctx, kv in shapes:
        kv = q + ctx if kv is None else kv
        R = q * G
        tiles = -(-R // PR)
        args = (R, q, kv, ctx, G, PR)
        pos = 0
        for t in range(tiles):
            last = min(PR * t + PR - 1, R - 1)
            keys = min(max(ctx + last // G + 1, 0), kv)
            n = max(1, -(-keys // 32))
            assert plan.chunks(*args, t) == n
            assert plan.prefix(*args, t) == pos, (args, t)
            pos += plan.tile_cost() + n
        assert plan.prefix(*args, tiles) == pos


@pytest.mark.parametrize("PR", [128, 192])
@pytest.mark.parametrize("G", [1, 3, 4, 5, 6, 7, 8, 10, 12, 24, 60, 63])
def test_long_prompts_take_a_few_steps(plan, G, PR):
    """Every tile of a long prompt costs the same few steps: a search over the tiles that walked
    them anew from the first would be quadratic in the prompt's length."""
    q, ctx = 32768 + 5, 1000
    R, kv = q * G, q + ctx
    tiles = -(-R // PR)
    args = (R, q, kv, ctx, G, PR)
    pos, want = 0, [0]
    for t in range(tiles):
        pos += plan.tile_cost() + -(-(ctx + (min(PR * (t + 1), R) - 1) // G + 1) // 32)
        want.append(pos)
    for t in [*range(0, tiles, max(1, tiles // 300)), tiles - 1, tiles]:
        plan.count()
        assert plan.prefix(*args, t) == want[t], t
        assert plan.count() <= 8, t
