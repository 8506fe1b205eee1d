"""Decode through whole-line K reads (up to 8 query rows per kv head) and past them: the short
decode of batches large enough to take them, with stale slots that hold NaN, at row counts on
both sides of 8, over 16-bit and E4M3 caches; and the stream-K decode on both sides of the unit
lengths where 16-bit and E4M3 caches take them, at row distances and query rows on both sides of theirs."""

from __future__ import annotations

import random

import pytest
import torch

from kvserve_amd import HipAttention, last_launch_kernels, last_launches, workloads
from oracle import fp8, torch_reference
from tests import paged_check as pc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(("heads", "q"), [((32, 8), 1), ((32, 8), 2), ((32, 8), 3), ((16, 16), 8), ((64, 8), 1)])
def test_short_decode(hip_device, heads, q, head_dim, e4m3):
    rng = random.Random(q)
    B = 64 if e4m3 else 40  # B Hkv D >= 16384; over E4M3 caches, D = 128, B Hkv D 1024 >= 48 Mi
    ctx = [0, 1, 7, 8, 15, 16, 17, 31, 32, 33, 40, 1024 - q] + [rng.randint(0, 700) for _ in range(B - 12)]
    w = workloads.custom("lines", [q] * B, ctx, *heads, head_dim, 16, seed=q)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=q)
    for t, n in zip(w.tables, w.seq_lens):  # slots past a sequence's keys hold anything
        if n % 16:
            b.k_cache[t[n // 16], n % 16 :] = float("nan")
            b.v_cache[t[n // 16], n % 16 :] = float("nan")
    if e4m3:
        k, v = fp8.quantize(b.k_cache, 1.0).to(hip_device), fp8.quantize(b.v_cache, 0.5).to(hip_device)
        HipAttention.write_kv(k, v, b.k_new, b.v_new, b.meta.slot_mapping, k_scale=1.0, v_scale=0.5)
        out = HipAttention.forward(b.q, k, v, b.meta, w.scale, k_scale=1.0, v_scale=0.5)
        kf, vf = fp8.dequantize(k.cpu(), 1.0), fp8.dequantize(v.cpu(), 0.5)
    else:
        out = pc.attend(b)
        kf, vf = b.k_cache.float().cpu(), b.v_cache.float().cpu()
    assert last_launch_kernels() == ["decode"]
    m = b.meta
    ref = torch_reference.forward(b.q.float().cpu(), kf.nan_to_num(), vf.nan_to_num(), m.block_tables.cpu(),
                                  m.seq_lens.cpu(), m.query_lens.cpu(), w.scale)  # fmt: skip
    assert (out.float().cpu() - ref).abs().max().item() <= pc.TOL_16BIT


@pytest.mark.parametrize("ctx", [4000, 4200, 12000])
@pytest.mark.parametrize(("heads", "q"), [((32, 8), 1), ((32, 8), 3), ((8, 1), 1)])
def test_stream_k_decode(hip_device, heads, q, ctx):
    # 128 units of 8-head groups: 32 sequences of 4096 keys give 32 chunks a unit
    B = 32 if heads[1] == 8 else 8
    lens = [ctx + 37 * i for i in range(B)] if ctx < 5000 else [ctx] + [200 + 61 * i for i in range(B - 1)]
    w = workloads.custom("stream", [q] * B, lens, *heads, 128, 16, seed=7)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=7)
    out = pc.attend(b)
    assert "reduce" in last_launch_kernels()
    assert pc.max_err_vs_oracle(b, out, [0, 1, B // 2, B - 1]) <= pc.TOL_16BIT


@pytest.mark.parametrize(("e4m3", "chunks"), [(False, 4), (False, 31), (False, 33), (True, 7), (True, 9)])
@pytest.mark.parametrize(("heads", "q", "head_dim"), [((32, 8), [1], 128), ((32, 8), [1, 2, 3], 128), ((24, 12), [4], 128),
                                                      ((16, 16), [1], 128), ((8, 2), [1], 128), ((32, 8), [1], 64)])  # fmt: skip
def test_stream_k_lines(hip_device, heads, q, head_dim, e4m3, chunks):
    """Sequences whose stale slots hold NaN, the mean unit about `chunks` chunks long; queries of 1 to 3 tokens
    make batches whose most query rows are past 8 while some sequences' are not."""
    H, Hkv = heads
    hgw = 8 if Hkv % 8 == 0 else 4 if Hkv % 4 == 0 else 2
    units = (2048 if e4m3 or head_dim == 64 else 1024) // hgw  # waves over heads a unit, on 256 CUs
    if e4m3 and head_dim == 64:
        units *= 2
    rng = random.Random(chunks)
    B = 20
    mean = chunks * units * 32 // (B * (Hkv // hgw))
    lens = [max(1, mean + rng.randint(-40, 40)) for _ in range(B)]
    if max(lens) + 4 <= 1024:
        lens[0] = 1100  # past the short decode
    w = workloads.custom("lines", [q[i % len(q)] for i in range(B)], lens, H, Hkv, head_dim, 16, seed=3)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=3)
    for t, n in zip(w.tables, w.seq_lens):
        if n % 16:
            b.k_cache[t[n // 16], n % 16 :] = float("nan")
            b.v_cache[t[n // 16], n % 16 :] = float("nan")
    out, kf, vf = _attend(b, e4m3)
    assert "reduce" in last_launch_kernels()
    _check(b, out, kf, vf, (0, 7, B - 1))


def _attend(b, e4m3):
    """The batch's attention, over the caches or over them in E4M3, and the values that they hold."""
    if not e4m3:
        return pc.attend(b), b.k_cache, b.v_cache
    k, v = ((x.float() / f).clamp(-448, 448).to(fp8.FP8) for x, f in ((b.k_cache, 1.0), (b.v_cache, 0.5)))
    HipAttention.write_kv(k, v, b.k_new, b.v_new, b.meta.slot_mapping, k_scale=1.0, v_scale=0.5)
    out = HipAttention.forward(b.q, k, v, b.meta, b.workload.scale, k_scale=1.0, v_scale=0.5)
    return out, k.float(), v.float() * 0.5


def _check(b, out, kf, vf, seqs):
    w = b.workload
    G, t0 = w.num_heads // w.num_kv_heads, 0
    for i, (n, s) in enumerate(zip(w.query_lens, w.seq_lens)):
        if i in seqs:
            rows = b.meta.block_tables[i, : -(-s // 16)]
            ks, vs = (x[rows].flatten(0, 1)[:s].float().repeat_interleave(G, 1) for x in (kf, vf))
            x = torch.einsum("qhd,khd->hqk", b.q[t0 : t0 + n].float().cpu(), ks.cpu()) * w.scale
            hidden = torch.arange(s)[None, :] > s - n + torch.arange(n)[:, None]
            ref = torch.einsum("hqk,khd->qhd", torch.softmax(x.masked_fill(hidden, float("-inf")), -1), vs.cpu())
            assert (out[t0 : t0 + n].float().cpu() - ref).abs().max().item() <= pc.TOL_16BIT
        t0 += n


@pytest.mark.parametrize("decodes", [6, 90])  # one launch with the chunk's tiles, a launch of their own
@pytest.mark.parametrize("e4m3", [False, True])
@pytest.mark.parametrize("q", [[1], [2], [1, 2, 4], [4]])
def test_beside_a_prompt_chunk(hip_device, q, e4m3, decodes):
    """Decoding sequences beside a prompt chunk, all of them up to 8 query rows, some, or none."""
    rng = random.Random(decodes)
    n = [q[i % len(q)] for i in range(decodes)]
    w = workloads.custom("beside", [*n, 130], [rng.randint(900, 1500) for _ in n] + [70], 32, 8, 128, 16, seed=4)
    b = workloads.materialize(w, torch.bfloat16, hip_device, seed=4)
    out, kf, vf = _attend(b, e4m3)
    assert last_launches() == (["mixed", "reduce"] if decodes == 6 else ["decode", "prefill", "reduce"])
    _check(b, out, kf, vf, (0, 1, 2, decodes - 1, decodes))
