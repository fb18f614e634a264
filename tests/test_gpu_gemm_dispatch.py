"""The bf16 product at the edges of its kernels' ranges, against the fp32
product of the same operands: K fp32 additions and one rounding to bf16, so at
most 2^-8 of a value and K 2^-24 of the sum of its terms' magnitudes."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1024, 2048, 192), (1408, 1536, 192),    # 512 and 528 tiles of 64 x 64
    (832, 2368, 2048), (1001, 2015, 128),    # 481 in one round with a long K; 512, the last ones cut
    (320, 320, 64), (4096, 4096, 64),        # the smallest K, and a full grid of 256 x 256
])
def test_product(m, n, k):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from gefen.kernels import _native
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, device="cuda", generator=gen).bfloat16()
    b = torch.randn(n, k, device="cuda", generator=gen).bfloat16()
    c = torch.randn(m, n, device="cuda", generator=gen).bfloat16()
    d = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    _native.check(_native.load().gefenx_gemm_nt_bf16(
        a.data_ptr(), b.data_ptr(), c.data_ptr(), d.data_ptr(), m, n, k, 0.5, -2.0,
        torch.cuda.current_stream().cuda_stream), "gemm")
    ref = 0.5 * (a.double() @ b.double().t()) - 2.0 * c.double()
    terms = 0.5 * (a.double().abs() @ b.double().abs().t()) + 2.0 * c.double().abs()
    assert ((d.double() - ref).abs() <= ref.abs() * 2.0 ** -8 + terms * (k + 2) * 2.0 ** -24).all()
