"""The per-step calls on tensors (_kvhtorch): plain valid calls are taken and give the bits of the
step-by-step path; everything else comes back as None and HipAttention raises (or computes) what it
does without them."""

from __future__ import annotations

import pytest
import torch

from kvserve_amd import HipAttention, _lib, workloads
from kvserve_amd.attention import FP8

pytestmark = pytest.mark.gpu


class _Sub(torch.Tensor):
    pass


@pytest.fixture
def batch(hip_device):
    w = workloads.custom("calls", [1, 3, 40], [30, 500, 7], 32, 8, 64, 16, seed=1)
    return workloads.materialize(w, torch.bfloat16, hip_device, seed=1)


def _args(b, **kw):
    a = {"q": b.q, "k": b.k_cache, "v": b.v_cache, "bt": b.meta.block_tables, "sl": b.meta.seq_lens,
         "qsl": b.meta.query_start_loc, "mq": b.meta.max_query_len, "scale": 0.125, "out": None, "ks": 1.0, "vs": 1.0}  # fmt: skip
    a.update(kw)
    return list(a.values())


def _without(monkeypatch, f):
    with monkeypatch.context() as m:
        m.setattr(_lib, "_calls", None)
        return f()


def test_taken_calls_give_the_same_bits(batch, monkeypatch):
    b, slots = batch, batch.meta.slot_mapping
    caches = [b.k_cache.clone(), b.v_cache.clone()]
    assert _lib.calls().write_kv(*caches, b.k_new, b.v_new, slots, 1.0, 1.0) is True
    _without(monkeypatch, lambda: HipAttention.write_kv(b.k_cache, b.v_cache, b.k_new, b.v_new, slots))
    assert torch.equal(caches[0], b.k_cache) and torch.equal(caches[1], b.v_cache)
    want = _without(monkeypatch, lambda: HipAttention.forward(b.q, b.k_cache, b.v_cache, b.meta, 0.125))
    got = _lib.calls().forward(*_args(b))
    assert torch.equal(got, want) and got.is_contiguous()
    wide = torch.zeros(b.q.shape[0], 40, 64, dtype=b.q.dtype, device=b.q.device)
    out = wide[:, 4:36]  # a strided output
    assert _lib.calls().forward(*_args(b, out=out)) is out and torch.equal(out, want)
    assert not wide[:, :4].any() and not wide[:, 36:].any()
    strided = torch.cat([b.q, b.q], dim=1)[:, :32]
    assert torch.equal(HipAttention.forward(strided, b.k_cache, b.v_cache, b.meta, 0.125), want)
    assert torch.equal(HipAttention.forward(b.q, b.k_cache, b.v_cache, b.meta, 0.125), want)


def test_refused_calls_are_left_to_the_method(batch):
    b = batch
    f = _lib.calls().forward
    assert f(*_args(b)) is not None
    fp8 = torch.zeros(b.k_cache.shape, dtype=torch.uint8, device=b.q.device).view(FP8)
    for kw in (
        {"q": b.q.float()}, {"q": b.q.cpu()}, {"q": b.q[..., ::2]}, {"q": b.q[0]}, {"q": b.q[:, :31]},
        {"k": b.k_cache.half()}, {"k": b.k_cache[:-1]}, {"k": fp8}, {"bt": b.meta.block_tables.int()},
        {"bt": b.meta.block_tables[:, ::2]}, {"sl": b.meta.seq_lens[:-1]}, {"qsl": b.meta.seq_lens},
        {"sl": b.meta.seq_lens.cpu()}, {"ks": 0.5}, {"out": b.q[:-1].clone()}, {"out": b.q.half()}, {"out": b.q.cpu()},
    ):  # fmt: skip
        assert f(*_args(b, **kw)) is None, kw.keys()
        a = dict(zip(("q", "k", "v", "bt", "sl", "qsl", "mq", "scale", "out", "ks", "vs"), _args(b, **kw)))
        meta = type(b.meta)(b.meta.slot_mapping, a["bt"], a["sl"], b.meta.query_lens, a["qsl"], b.meta.max_seq_len, a["mq"])
        with pytest.raises(ValueError):
            HipAttention.forward(a["q"], a["k"], a["v"], meta, a["scale"], a["out"], a["ks"], a["vs"])
    for s in (0.0, -1.0, float("inf"), float("nan")):
        assert f(*_args(b, k=fp8, v=fp8, ks=s)) is None
    assert f(*_args(b, k=fp8, v=fp8, ks=2.0, vs=0.5)) is not None
    # no plain tensor or number: left to the method, which takes them
    assert f(*_args(b, q=b.q.as_subclass(_Sub))) is None
    assert f(*_args(b, scale=torch.tensor(0.125))) is None
    assert f(*_args(b, mq=True)) is None
    w = _lib.calls().write_kv
    slots = b.meta.slot_mapping
    assert w(b.k_cache, b.v_cache, b.k_new, b.v_new, slots, 1.0, 1.0) is True
    for bad in (
        (b.k_cache, b.v_cache, b.k_new[:-1], b.v_new, slots), (b.k_cache, b.v_cache, b.k_new, b.v_new, slots[:-1]),
        (b.k_cache, b.v_cache, b.k_new.half(), b.v_new.half(), slots), (b.k_cache, b.v_cache, b.k_new, b.v_new, slots.int()),
        (b.k_cache.cpu(), b.v_cache.cpu(), b.k_new, b.v_new, slots),
    ):  # fmt: skip
        assert w(*bad, 1.0, 1.0) is None
        with pytest.raises(ValueError):
            HipAttention.write_kv(*bad)


def test_status_errors_still_raise(batch):
    b = batch
    q = torch.cat([b.q.flatten(), b.q.flatten()])[1 : 1 + b.q.numel()].view(b.q.shape)  # 2 bytes off: KVH_E_ALIGN
    with pytest.raises(_lib.KvhError, match="kvh_paged_attention.*aligned"):
        HipAttention.forward(q, b.k_cache, b.v_cache, b.meta, 0.125)
