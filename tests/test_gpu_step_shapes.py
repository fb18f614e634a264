"""The step kernels at the edges of their variants, against the oracle.

Each case is one tensor (shape, block length, dtype, layout, rounding) with a
preset period and the golden codebook, stepped from zero state, alone and in one
launch with a larger companion.  Small launches cut the stats into granules and
the apply into short tasks whatever the companion here is; the cases of
test_large_launch stand beside so much else that they take whole tiles and long
tasks.  Checked against the oracle's step: indices and magnitudes bit-exact, v
within 1e-6 relative, parameters within 1 ulp (fp32: 1e-6 relative).
"""
from __future__ import annotations

import ctypes
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


def _golden_codebook():
    return torch.from_numpy(np.load(os.path.join(GOLD, "learn.npz"))["cb"]).float()


def _data(shape, dtype, layout, dev, seed, scale, plant=None):
    """The same values whatever the layout; companions of millions of elements
    are made on the device."""
    if layout.startswith("big"):
        return torch.full(shape[::-1], scale, dtype=dtype, device=dev).t() if layout == "big-t" else \
            torch.full(shape, scale, dtype=dtype, device=dev)
    t = _values(shape, dtype, torch.Generator().manual_seed(seed), scale)
    return _place(plant(t) if plant else t, layout, dev)


def _steps(dev, specs, kw, cb=None, steps=SEED_STEPS, plants={}):
    """Step the tensors of `specs` together; per step the optimizer's state.
    plants: by step, what is done to the first tensor's grad."""
    from gefen import Gefen
    cb = _golden_codebook() if cb is None else cb
    params = [torch.nn.Parameter(_data(shape, dtype, layout, dev, 11 + i, 0.02))
              for i, (shape, period, dtype, layout) in enumerate(specs)]
    opt = Gefen([("p%d" % i, p) for i, p in enumerate(params)], lr=LR, weight_decay=WD,
                factored_v_2d=kw.get("factored", True), stochastic_round=kw.get("sr", False))
    opt._gefen_codebook = cb.to(dev)
    for p, (_, period, _, _) in zip(params, specs):
        opt.state[p]["automatic_period"] = period
    out = []
    for s in range(steps):
        for i, (p, (shape, _, dtype, layout)) in enumerate(zip(params, specs)):
            p.grad = _data(shape, dtype, layout, dev, 1000 * (s + 1) + i, 1e-3, plants.get(s) if i == 0 else None)
        opt.step()
        torch.cuda.synchronize()
        st = opt.state[params[0]]
        out.append({"p": params[0].detach().float().cpu().numpy().copy(),
                    **{k: st[k].cpu().numpy().reshape(-1).copy()
                       for k in ("m_codebook", "m_magnitude", "v_row", "v_col", "vmean") if k in st}})
    return out, cb.numpy()


def _id(c):
    return "%s-P%d-%s-%s%s" % ("x".join(map(str, c[0])), c[1], str(c[2])[6:], c[3], "".join("-" + k for k in c[4]))


def _check(dev, case, companions, cb=None, steps=SEED_STEPS, plants={}):
    shape, period, dtype, layout, kw = case
    got, cb = _steps(dev, [(shape, period, dtype, layout)] + companions, kw, cb, steps, plants)
    code = TDT_CODE[dtype]
    factored = len(shape) == 2 and kw.get("factored", True)
    n = int(np.prod(shape))
    p = _values(shape, dtype, torch.Generator().manual_seed(11), 0.02).float().numpy()
    idx, mag = np.zeros(n, np.uint8), np.zeros(n // period, np.float32)
    v = [np.zeros(shape[0], np.float32), np.zeros(shape[-1], np.float32)] if factored else \
        [np.zeros(n // period, np.float32)]
    for s in range(steps):
        g = _values(shape, dtype, torch.Generator().manual_seed(1000 * (s + 1)), 1e-3)
        g = (plants[s](g) if s in plants else g).float().numpy()
        args = dict(beta1=0.9, beta2=0.999, lr=LR, eps=1e-8, bc1=1 - 0.9 ** (s + 1), bc2=1 - 0.999 ** (s + 1), wd=WD,
                    sr_seed=s if kw.get("sr") else None)
        if factored:
            p, idx, mag, v[0], v[1] = orc.factored_step(p, g, idx, mag, v[0], v[1], period, cb, code, **args)
        else:
            p, idx, mag, v[0] = orc.block_step(p, g, idx, mag, v[0], period, cb, code, **args)
        tag = "%s step %d" % (case, s + 1)
        np.testing.assert_array_equal(got[s]["m_magnitude"], mag, err_msg=tag)
        assert np.array_equal(got[s]["m_codebook"], idx), tag
        for key, ref in zip(("v_row", "v_col") if factored else ("vmean",), v):
            np.testing.assert_allclose(got[s][key], ref, rtol=1e-6, atol=0, err_msg=tag)
        if not plants:
            assert_within_ulp(got[s]["p"], p, code, tag, atol=1e-6 * LR)
        p = got[s]["p"].reshape(shape)  # the next step from the same parameters: one step's rounding at a time


@pytest.mark.parametrize("companion", [None, (1500, 1024)])
@pytest.mark.parametrize("case", CASES, ids=_id)
def test_step_matches_oracle(dev, case, companion):
    _check(dev, case, [(companion, companion[1], case[2], "c")] if companion else [])


# whole tiles: several granules, the last cut by the last row (views: column);
# tasks of 8 row steps with a cut last task (the aligned kernel and the any-width
# one; several rows to a step)
LARGE = [
    ((257, 1024), 1024, BF16, "c", {}),
    ((1501, 2048), 2048, F16, "c", {}),
    ((301, 2056), 2056 * 301, F32, "c", {}),
    ((300, 1025), 1025, BF16, "o", {}),
    ((333, 768), 24, BF16, "c", {"sr": True}),
    ((9000, 16), 48, BF16, "c", {}),
    ((4099, 33), 4099, BF16, "c", {}),
    ((2100, 250), 250, F16, "o", {}),
    ((256, 256), 256, BF16, "t", {}),
    ((264, 1096), 1096, BF16, "t", {}),
    ((1000, 1800), 1800, F16, "t", {}),
]


def _granule_bytes(specs):
    """What the launches of these tensors take for granules as workgroups."""
    from gefen.kernels import _native
    lib = _native.load()
    code = {F32: _native.DT_F32, F16: _native.DT_F16, BF16: _native.DT_BF16}
    d = (_native.TensorDesc * len(specs))()
    for x, (shape, period, dtype, layout) in zip(d, specs):
        for f in ("p", "grad", "m_codebook", "m_magnitude", "v0", "v1", "workspace"):
            setattr(x, f, 4096 + (2 if layout == "o" else 0))
        x.rows, x.cols, x.period, x.dtype, x.factored = shape[0], shape[1], period, code[dtype], 1
        x.ps0 = x.gs0 = 1 if layout.endswith("t") else shape[1]
        x.ps1 = x.gs1 = shape[0] if layout.endswith("t") else 1
    return lib.gefenx_multi_tensor_scratch_bytes_for(ctypes.addressof(d), len(specs)) - \
        lib.gefenx_multi_tensor_scratch_bytes(len(specs))


@pytest.mark.parametrize("case", LARGE, ids=_id)
def test_large_launch(dev, case):
    """Beside 67M elements (views: 1.1e9) of its own kernel: the launch takes
    whole tiles, where alone it takes granules."""
    spec = case[:4]
    big = ((16384, 65536), 65536, case[2], "big-t") if case[3] == "t" else ((16384, 4096), 4096, case[2], "big")
    assert _granule_bytes([spec]) > 0
    assert _granule_bytes([spec, big]) == _granule_bytes([big])
    _check(dev, case, [big])


def _dense_codebook():
    """Many codewords within 1/2048 of each other, equal ones among them, near
    zero, at a quarter and at the end."""
    cb = torch.cat([torch.linspace(-1, 1, 96), torch.linspace(-0.003, 0.003, 56), torch.linspace(0.25, 0.2503, 40),
                    torch.full((24,), -0.125), torch.linspace(0.9997, 1, 40)])
    return torch.sort(cb)[0].contiguous()


@pytest.mark.parametrize("case", CASES, ids=_id)
def test_dense_codebook(dev, case):
    _check(dev, case, [], cb=_dense_codebook(), steps=3)


@pytest.mark.parametrize("kind", ["nan", "inf", "huge"])
@pytest.mark.parametrize("case", CASES, ids=_id)
def test_nonfinite_grads(dev, case, kind):
    """Magnitudes (torch's amax: NaN above inf), indices and v where grads of the
    second step hold NaN, infinities, or values whose squares overflow, in the
    first and the last element, beside chunk borders and in the last column; the
    third step has the state that they left."""
    def plant(g):
        big = 6e4 if g.dtype == F16 else 1e20
        a, b = {"nan": (float("nan"), float("nan")), "inf": (float("inf"), -float("inf")), "huge": (big, -big)}[kind]
        x, c = g.clone().reshape(-1), g.shape[-1]
        n = x.numel()
        x[0], x[n - 1], x[n // 2 // c * c + c - 1] = a, b, b
        x[min(n // 3 // 8 * 8 + 7, n - 1)] = a
        x[min(n // 5 // 8 * 8, n - 1)] = b
        return x.reshape(g.shape)
    _check(dev, case, [], steps=3, plants={1: plant})
