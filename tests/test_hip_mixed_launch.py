"""Batches with prompt chunks: decode and prefill units in one launch (small decode parts) against
the same batch in two launches (as when the call's kernels are timed), and against the oracle.
Shapes: prompts alone, decodes between them, more sequences than a workgroup has threads (each
thread then plans several), tiles on both sides of a tile's last row, GQA groups that do not
divide a tile."""

from __future__ import annotations

import ctypes
import random

import pytest
import torch

from kvserve_amd import _lib, last_launch_kernels, workloads
from tests import paged_check as pc

pytestmark = pytest.mark.gpu


def _apart(batch) -> torch.Tensor:
    """The batch's attention with the timing hook armed."""
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(5)]
    for e in ev:
        e.record()
    handles = (ctypes.c_void_p * 5)(*[e.cuda_event for e in ev])
    _lib.check(_lib.load().kvh_profile_arm(handles, 5), "kvh_profile_arm")
    return pc.attend(batch, write=False)


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
    raise ValueError(name)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("name", ["prompts", "between_decodes", "many_sequences", "group_of_5"])
def test_one_launch_equals_two(hip_device, name, head_dim):
    q, ctx, (H, Hkv) = _shape(name)
    w = workloads.custom(name, q, ctx, H, Hkv, head_dim, 16, seed=3)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=3)
    out = pc.attend(b)
    assert last_launch_kernels() == ["decode", "prefill", "reduce"]
    assert torch.equal(out, _apart(b))  # the same tiles, pieces and merge order
    seqs = list(range(len(q))) if len(q) < 50 else list(range(0, len(q), 7))
    assert pc.max_err_vs_oracle(b, out, seqs, rows_per_seq=12) <= pc.TOL_16BIT
