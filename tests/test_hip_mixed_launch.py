"""Batches with prompt chunks: decode and prefill units in one launch (small decode parts) against the
same batch in two launches (its block tables widened, so that the decode part could be large), and against
the oracle. Shapes: prompts alone, decodes between them, more sequences than a workgroup has threads (each
thread then plans several), tiles on both sides of a tile's last row, GQA groups that do not divide a tile,
a long prompt of such a group, decode parts on both sides of the line between one launch and two."""

from __future__ import annotations

import ctypes
import random
from dataclasses import replace

import pytest
import torch

from kvserve_amd import HipAttention, _lib, last_launch_kernels, last_launches, workloads
from oracle import fp8
from tests import paged_check as pc

pytestmark = pytest.mark.gpu


def _shape(name: str) -> tuple[list[int], list[int], tuple[int, int]]:
    rng = random.Random(name)
    if name == "prompts":
        return [700, 48, 49, 191, 1], [0, 31, 32, 500, 0], (32, 8)
    if name == "between_decodes":
        return [1, 130, 1, 1, 97, 2, 300], [40, 0, 17, 3, 900, 64, 5], (32, 8)
    if name == "many_sequences":  # 300 sequences: two per planning thread
        q = [rng.choice([1, 1, 1, 17, 33]) for _ in range(300)]
        return q, [rng.randint(0, 60) for _ in q], (8, 4)
    if name == "group_of_5":
        return [80, 1, 39, 200], [10, 20, 0, 333], (10, 2)
    if name == "long_group_of_7":  # 300 16-bit tiles: units start in every window of the tile search
        return [8200, 1, 70], [30, 20, 5], (7, 1)
    raise ValueError(name)


def _forward(b, caches=None, meta=None) -> torch.Tensor:
    meta = meta or b.meta
    if caches is None:
        return HipAttention.forward(b.q, b.k_cache, b.v_cache, meta, b.workload.scale)
    return HipAttention.forward(b.q, *caches, meta, b.workload.scale, k_scale=1.0, v_scale=0.5)


def _e4m3(b):
    """The batch's caches in E4M3, and the batch holding their values for the oracle."""
    caches = [(x.float() / f).clamp(-448, 448).to(fp8.FP8) for x, f in ((b.k_cache, 1.0), (b.v_cache, 0.5))]
    HipAttention.write_kv(*caches, b.k_new, b.v_new, b.meta.slot_mapping, k_scale=1.0, v_scale=0.5)
    return caches, replace(b, k_cache=caches[0].float(), v_cache=caches[1].float() * 0.5)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("name", ["prompts", "between_decodes", "many_sequences", "group_of_5", "long_group_of_7"])
def test_one_launch_equals_two(hip_device, name, e4m3, head_dim):
    q, ctx, (H, Hkv) = _shape(name)
    w = workloads.custom(name, q, ctx, H, Hkv, head_dim, 16, seed=3)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=3)
    HipAttention.write_kv(b.k_cache, b.v_cache, b.k_new, b.v_new, b.meta.slot_mapping)
    caches, ref = _e4m3(b) if e4m3 else (None, b)
    out = _forward(b, caches)
    assert last_launches() == ["mixed", "reduce"]
    assert last_launch_kernels() == ["decode", "prefill", "reduce"]
    wide = torch.zeros((len(q), 32768), dtype=torch.int64, device=hip_device)
    wide[:, : b.meta.block_tables.shape[1]] = b.meta.block_tables
    apart = _forward(b, caches, replace(b.meta, block_tables=wide))
    assert last_launches() == ["decode", "prefill", "reduce"]
    if name == "long_group_of_7":  # as many units as the launch's kernel holds: other pieces
        assert (out.float() - apart.float()).abs().max().item() <= pc.TOL_16BIT
    else:
        assert torch.equal(out, apart)  # the same tiles, pieces and merge order
    seqs = list(range(len(q))) if len(q) < 50 else list(range(0, len(q), 7))
    assert pc.max_err_vs_oracle(ref, out, seqs, rows_per_seq=12) <= pc.TOL_16BIT


@pytest.mark.parametrize(("e4m3", "decodes", "launches"), [
    (False, 9, ["mixed", "reduce"]), (False, 16, ["mixed", "reduce"]), (False, 17, ["decode", "prefill", "reduce"]),
    (True, 20, ["mixed", "reduce"]), (True, 32, ["mixed", "reduce"]), (True, 33, ["decode", "prefill", "reduce"]),
])  # fmt: skip
def test_decode_part_at_the_line(hip_device, e4m3, decodes, launches):
    """32 chunks a sequence over 128 units (256 over E4M3 caches): at most 4 chunks a unit share a launch, from 2
    on more than every unit's least, so the split is capped."""
    w = workloads.custom("line", [1] * decodes + [200], [1000] * decodes + [50], 32, 8, 128, 16, seed=5)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=5)
    HipAttention.write_kv(b.k_cache, b.v_cache, b.k_new, b.v_new, b.meta.slot_mapping)
    caches, ref = _e4m3(b) if e4m3 else (None, b)
    out = _forward(b, caches)
    assert last_launches() == launches
    assert pc.max_err_vs_oracle(ref, out, [0, 1, decodes // 2, decodes - 1, decodes], rows_per_seq=12) <= pc.TOL_16BIT


@pytest.mark.parametrize("decodes", [3, 17])  # one launch, two launches
def test_timing_changes_nothing(hip_device, decodes):
    """The timing hook times the launches that run without it: the same kernels, one event after each, the same
    bits."""
    w = workloads.custom("timed", [1] * decodes + [200, 90], [1000] * decodes + [50, 0], 32, 8, 128, 16, seed=5)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=5)
    out = pc.attend(b)
    launches = last_launches()
    assert launches == (["mixed", "reduce"] if decodes == 3 else ["decode", "prefill", "reduce"])
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(5)]
    for e in ev:
        e.record()
    handles = (ctypes.c_void_p * 5)(*[e.cuda_event for e in ev])
    _lib.check(_lib.load().kvh_profile_arm(handles, 5), "kvh_profile_arm")
    timed = pc.attend(b, write=False)
    assert last_launches() == launches and torch.equal(out, timed)
    torch.cuda.synchronize()
    # event k follows launch k, which takes microseconds: none is recorded twice around nothing
    assert all(ev[k].elapsed_time(ev[k + 1]) > 1e-3 for k in range(len(launches)))
