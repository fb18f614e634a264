"""A matrix that carries `placements`, as sharded parameters do, keeps the
block-shared second moment, a plain nn.Parameter with the attribute included."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_parameter_with_placements_takes_the_block_path():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from gefen import Gefen
    params = [torch.nn.Parameter(torch.randn(64, 64, device="cuda")) for _ in range(2)]
    params[1].placements = ("Shard(0)",)
    for p in params:
        p.grad = torch.randn_like(p)
    opt = Gefen([("p%d" % i, p) for i, p in enumerate(params)], lr=1e-3)
    opt.step()
    assert "v_row" in opt.state[params[0]] and "vmean" not in opt.state[params[0]]
    assert "vmean" in opt.state[params[1]] and "v_row" not in opt.state[params[1]]
