"""The step kernels at the edges of their variants, against the oracle.

Each case is one tensor (shape, block length, dtype, layout, rounding) with a
preset period and the golden codebook, stepped twice from zero state, alone
and in one launch with a larger companion (the stats tiles depend on the
launch's size).  Checked against the oracle's step: indices and magnitudes
bit-exact, v within 1e-6 relative, parameters within 1 ulp (fp32: 1e-6
relative).
"""
from __future__ import annotations

import os

import numpy as np
import pytest
import torch

from local_checks import TDT_CODE, assert_within_ulp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16
LR, WD, SEED_STEPS = 1e-3, 0.01, 2

# shape, period, dtype, layout ("c" contiguous, "t" transposed view, "o" an
# element offset into a flat buffer), options
CASES = [
    # stats tiles: rows around the 32-row granule, columns around a tile
    ((31, 1024), 1024, BF16, "c", {}),
    ((33, 1032), 1032, BF16, "c", {}),
    ((257, 2056), 2056 * 257, F32, "c", {}),
    ((520, 1024), 4096, F16, "c", {}),
    # transposed views: bands and column tiles
    ((256, 64), 64, BF16, "t", {}),
    ((264, 1096), 1096, BF16, "t", {}),
    ((1000, 200), 1600, F16, "t", {"factored": False}),
    # contiguous stats of any width: chunks cut by the last column, blocks that
    # end inside a chunk, storage that starts between vectors
    ((70, 1025), 1025, BF16, "c", {}),
    ((64, 1539), 3, F16, "c", {}),
    ((65, 771), 771 * 5, F32, "c", {}),
    ((40, 1031), 1031 * 4, BF16, "o", {}),
    ((96, 1024), 24, BF16, "o", {}),
    ((129, 520), 8, F32, "c", {}),
    # lane tiles: 1 to 64 lanes per row, a cut chunk, several tiles, blocks of
    # any length in a wave
    ((9, 8), 8, F32, "c", {}),
    ((3000, 16), 48, BF16, "c", {}),
    ((1025, 13), 65, F16, "c", {}),
    ((515, 250), 250, BF16, "o", {}),
    ((4099, 33), 4099, BF16, "c", {}),
    ((300, 256), 300 * 256, F32, "c", {}),
    ((70, 1100), 100, BF16, "c", {}),
    ((96, 1031), 96, F16, "c", {}),
    ((64, 512), 8, BF16, "c", {}),
    ((66, 2048), 1, F32, "c", {}),
    ((48, 600), 72, BF16, "t", {}),
    # apply: segments of any width, chunks that hold a block border, a task's
    # rows cut by the last row, stochastic rounding, the flat walk's last chunk
    ((9, 513), 513, BF16, "c", {}),
    ((17, 1543), 1543 * 17, F16, "o", {}),
    ((24, 1030), 10, BF16, "c", {}),
    ((45, 768), 9, F32, "o", {}),
    ((20, 16392), 16392, BF16, "c", {}),
    ((33, 1025), 1025, BF16, "c", {"sr": True}),
    ((50, 40), 8, F32, "c", {"sr": True}),
    ((64, 1024), 2048, F16, "c", {"sr": True}),
    ((41, 1031), 1031, BF16, "c", {"factored": False}),
    ((41, 1031), 1031, F16, "o", {"factored": False, "sr": True}),
    ((4097 * 9,), 9, F32, "c", {}),
    ((999,), 27, BF16, "c", {}),
    ((3047,), 277, F16, "c", {}),
    ((2048 * 11 + 8,), 8, BF16, "o", {}),
    # fewer than 8 columns: element loads
    ((500, 7), 35, BF16, "c", {}),
]


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.device("cuda", 0)


def _place(t, layout, dev):
    if layout == "t":
        return t.t().contiguous().to(dev).t()
    if layout == "o":  # the storage starts one element into an allocation
        flat = torch.zeros(t.numel() + 9, dtype=t.dtype, device=dev)
        flat[1:1 + t.numel()].copy_(t.reshape(-1))
        return flat[1:1 + t.numel()].view(t.shape)
    return t.to(dev)


def _values(shape, dtype, gen, scale):
    return (torch.randn(*shape, generator=gen) * scale).to(dtype)


def _steps(dev, specs, kw):
    """Step the tensors of `specs` together; per step the optimizer's state."""
    from gefen import Gefen
    cb = torch.from_numpy(np.load(os.path.join(GOLD, "learn.npz"))["cb"]).float()
    params = []
    for i, (shape, period, dtype, layout) in enumerate(specs):
        gen = torch.Generator().manual_seed(11 + i)
        params.append(torch.nn.Parameter(_place(_values(shape, dtype, gen, 0.02), layout, dev)))
    opt = Gefen([("p%d" % i, p) for i, p in enumerate(params)], lr=LR, weight_decay=WD,
                factored_v_2d=kw.get("factored", True), stochastic_round=kw.get("sr", False))
    opt._gefen_codebook = cb.to(dev)
    for p, (_, period, _, _) in zip(params, specs):
        opt.state[p]["automatic_period"] = period
    out = []
    for s in range(SEED_STEPS):
        for i, (p, (shape, _, dtype, layout)) in enumerate(zip(params, specs)):
            gen = torch.Generator().manual_seed(1000 * (s + 1) + i)
            p.grad = _place(_values(shape, dtype, gen, 1e-3), layout, dev)
        opt.step()
        torch.cuda.synchronize()
        st = opt.state[params[0]]
        out.append({"p": params[0].detach().float().cpu().numpy().copy(),
                    **{k: st[k].cpu().numpy().reshape(-1).copy()
                       for k in ("m_codebook", "m_magnitude", "v_row", "v_col", "vmean") if k in st}})
    return out, cb.numpy()


@pytest.mark.parametrize("companion", [None, (1500, 1024)])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%s-P%d-%s-%s%s" % (
    "x".join(map(str, c[0])), c[1], str(c[2])[6:], c[3], "".join("-" + k for k in c[4])))
def test_step_matches_oracle(dev, case, companion):
    shape, period, dtype, layout, kw = case
    specs = [(shape, period, dtype, layout)]
    if companion:
        specs.append((companion, companion[1], dtype, "c"))
    got, cb = _steps(dev, specs, kw)
    code = TDT_CODE[dtype]
    factored = len(shape) == 2 and kw.get("factored", True)
    n = int(np.prod(shape))
    p = _values(shape, dtype, torch.Generator().manual_seed(11), 0.02).float().numpy()
    idx, mag = np.zeros(n, np.uint8), np.zeros(n // period, np.float32)
    v = [np.zeros(shape[0], np.float32), np.zeros(shape[-1], np.float32)] if factored else \
        [np.zeros(n // period, np.float32)]
    for s in range(SEED_STEPS):
        g = _values(shape, dtype, torch.Generator().manual_seed(1000 * (s + 1)), 1e-3).float().numpy()
        args = dict(beta1=0.9, beta2=0.999, lr=LR, eps=1e-8, bc1=1 - 0.9 ** (s + 1), bc2=1 - 0.999 ** (s + 1), wd=WD,
                    sr_seed=s if kw.get("sr") else None)
        if factored:
            p, idx, mag, v[0], v[1] = orc.factored_step(p, g, idx, mag, v[0], v[1], period, cb, code, **args)
        else:
            p, idx, mag, v[0] = orc.block_step(p, g, idx, mag, v[0], period, cb, code, **args)
        tag = "%s step %d" % (case, s + 1)
        assert np.array_equal(got[s]["m_magnitude"], mag), tag
        assert np.array_equal(got[s]["m_codebook"], idx), tag
        for key, ref in zip(("v_row", "v_col") if factored else ("vmean",), v):
            np.testing.assert_allclose(got[s][key], ref, rtol=1e-6, atol=0, err_msg=tag)
        assert_within_ulp(got[s]["p"], p, code, tag, atol=1e-6 * LR)
        p = got[s]["p"].reshape(shape)  # the next step from the same parameters: one step's rounding at a time
