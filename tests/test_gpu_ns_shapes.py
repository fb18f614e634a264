"""Newton-Schulz on shapes around the 64-wide padding of its buffers, against
the oracle: relative Frobenius error <= 2e-2 (the reference's own
batched-vs-serial bound; the GEMMs accumulate in fp32 in another order)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
TUNED3 = [(5.0067, -14.4125, 10.6001), (3.7534, -6.8083, 3.3840), (3.2080, -4.3501, 2.0330)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [(1, 9), (63, 65), (64, 64), (65, 129), (130, 40), (200, 333), (511, 257),
                                   (300, 1030), (1408, 1409), (1700, 900)])
def test_shapes_around_the_padding(shape, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from gefen.gefen_muon import _zeropower_via_newtonschulz_batched as ns
    gen = torch.Generator().manual_seed(shape[0] * 1000 + shape[1])
    # three matrices, so the later ones start at any element alignment
    x = (torch.randn(3, *shape, generator=gen) * 1e-3).to(dtype)
    got = ns(x.cuda(), TUNED3, 3, 1e-7).float().cpu().numpy()
    for i in range(3):
        ref = orc.newton_schulz(x[i].float().numpy(), TUNED3)
        err = np.linalg.norm(got[i] - ref) / np.linalg.norm(ref)
        assert err <= 2e-2, (shape, dtype, i, err)


def test_non_finite_matrix_stays_non_finite():
    """A NaN or inf entry reaches every entry of the result, as unpadded."""
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from gefen.gefen_muon import _zeropower_via_newtonschulz_batched as ns
    x = torch.randn(2, 70, 100, generator=torch.Generator().manual_seed(3))
    x[0, 5, 7] = float("nan")
    x[1, 69, 99] = float("inf")
    assert torch.isnan(ns(x.cuda(), TUNED3, 3, 1e-7)).all()
