"""The skinny GEMM's forms (csrc/skinny.h) at the sizes where they change or end: 8192 weight rows
(x staged in LDS), 8 / 9, 16 / 17, 32 / 33 and 64 rows of x, rows that leave a workgroup's last
tiles empty, one and several chunks of k; against an fp32 product, and the fused SiLU * up bit for
bit against the two steps."""

from __future__ import annotations

import pytest
import torch

from kvserve_amd import _lib
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
