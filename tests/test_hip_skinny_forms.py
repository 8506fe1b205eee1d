"""The skinny GEMM's forms (csrc/skinny.h) at the sizes where they change or end: 8192 weight rows
(x staged in LDS), 8 / 9, 16 / 17, 32 / 33 and 64 rows of x, rows that leave a workgroup's last
tiles empty, one and several chunks of k; against an fp32 product, and the fused SiLU * up bit for
bit against the two steps."""

from __future__ import annotations

import pytest
import torch

from kvserve_amd import HipAttention, _lib
from kvserve_amd.engine import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [5, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize(("n", "k"), [(8176, 1024), (8192, 1024), (8208, 2048), (16400, 3072)])
def test_gemm_skinny_forms(hip_device, m, n, k):
    g = torch.Generator(device=hip_device).manual_seed(m * n)
    x = torch.randn(m, k, generator=g, device=hip_device).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device=hip_device) / k**0.5).to(torch.bfloat16)
    got = ops.gemm_skinny(x, w)
    want = x.float() @ w.float().t()
    # one rounding to bf16 (2^-8 of the value at most) over sums of O(1) terms kept in fp32
    torch.testing.assert_close(got.float(), want, rtol=2**-8, atol=1e-4)
    assert torch.equal(got, ops.gemm_skinny(x, w))
    y = torch.empty((m, n // 2), dtype=x.dtype, device=hip_device)
    st = _lib.load().kvh_gemm_skinny_silu_mul(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(),
                                              y.stride(0), m, n // 2, k, _lib.KVH_DTYPE[x.dtype],
                                              torch.cuda.current_stream().cuda_stream)  # fmt: skip
    _lib.check(st, "kvh_gemm_skinny_silu_mul")
    assert torch.equal(y, ops.silu_mul(got))
    # rows 2 bytes off the 8-byte grid take the narrow stores
    z = torch.empty((m, n + 1), dtype=x.dtype, device=hip_device)[:, :n]
    st = _lib.load().kvh_gemm_skinny(x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), z.data_ptr(), z.stride(0),
                                     m, n, k, _lib.KVH_DTYPE[x.dtype], torch.cuda.current_stream().cuda_stream)  # fmt: skip
    _lib.check(st, "kvh_gemm_skinny")
    assert torch.equal(z, got)


@pytest.mark.parametrize("m", [5, 8, 9, 17, 33, 48, 49])
@pytest.mark.parametrize(("n", "k"), [(2048, 1024), (2048, 2048), (2064, 2048), (5104, 2048), (5120, 1024), (5120, 2048),
                                      (8192, 2048), (8208, 1024), (10240, 2048), (12304, 1024), (16400, 1024)])  # fmt: skip
def test_lines_between_forms(hip_device, m, n, k):
    """Both sides of the lines that rows of the weight, k and rows of x draw between the forms, fused with RoPE
    and the cache write (the same bits as the projection and the separate step) and alone."""
    g = torch.Generator(device=hip_device).manual_seed(m * n + k)
    x = torch.randn(m, k, generator=g, device=hip_device).to(torch.bfloat16)
    w = (torch.randn(n, k, generator=g, device=hip_device) / k**0.5).to(torch.bfloat16)
    got = ops.gemm_skinny(x, w)
    torch.testing.assert_close(got.float(), x.float() @ w.float().t(), rtol=2**-8, atol=1e-4)
    D, Hkv = 16, 1  # heads of 16: any n of this list is (H + 2) heads
    H = n // D - 2 * Hkv
    cos = torch.rand(64, D, generator=g, device=hip_device)
    sin = torch.rand(64, D, generator=g, device=hip_device)
    pos = torch.arange(m, device=hip_device)
    kv = [torch.zeros(4, 16, Hkv, D, dtype=torch.bfloat16, device=hip_device) for _ in range(4)]
    q = HipAttention.gemv_rope_and_cache(x, w, pos, cos, sin, kv[0], kv[1], pos, H)
    want = HipAttention.rope_and_cache(got, pos, cos, sin, kv[2], kv[3], pos, H)
    assert torch.equal(q, want) and torch.equal(kv[0], kv[2]) and torch.equal(kv[1], kv[3])
