"""A tensor's factored step does not depend on what else a call holds, on how
much scratch it is given, or on the entry point: the same bits of every output.

The gradients make the order of the float64 additions decide an fp32 rounding.
A column (of a view, a row) holds 2^60 and 2^36, whose sum lies halfway between
two fp32 values, and squares of 2^4 that are lost when added to it one group at
a time and are not when they meet each other first; so sums cut at another row
or column come out an fp32 ulp (2^-23) apart, far above what the float64
additions themselves are off (n 2^-53).
"""
from __future__ import annotations

import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16

# shape, period, dtype, transposed view, first and last row (views: column) of the small values
CASES = [
    ((2048, 1024), 1024, BF16, False, (32, 64)),
    ((2048, 1024), 2048 * 1024, F32, False, (32, 64)),
    ((4099, 1031), 1031, BF16, False, (32, 64)),
    ((2048, 512), 256, BF16, False, (32, 64)),          # lane tiles: short blocks
    ((65536, 16), 16, F32, False, (1024, 2048)),        # narrow: 1024 rows to a granule
    ((256, 4096), 4096, BF16, True, (64, 256)),
    ((2048, 1023), 1023, BF16, True, (32, 64)),         # a view the general kernels take
]


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.device("cuda", 0)


def _grad(shape, dtype, view, span):
    """Every other column (of a view, row) holds the values; the rest are zero."""
    g = torch.zeros(shape, dtype=torch.float32)
    tv = view and shape[0] % 8 == 0 and shape[1] % 8 == 0
    x = g.t() if tv else g
    lo, hi = span
    x[0, ::2], x[8 if tv else 1, ::2] = 2.0 ** 30, 2.0 ** 18  # in different fp32 partial sums
    x[lo:hi:8 if tv else 1, ::2] = 4.0
    return g.to(dtype)


def _place(t, view, dev):
    return t.t().contiguous().to(dev).t() if view else t.to(dev)


def _codebook(dev):
    return torch.from_numpy(np.load(os.path.join(GOLD, "learn.npz"))["cb"]).float().to(dev)


def _step(dev, case, companions):
    """One step of the case's tensor beside others: its parameter and state."""
    from gefen import Gefen
    shape, period, dtype, view, span = case
    p = torch.nn.Parameter(_place(torch.zeros(shape, dtype=dtype), view, dev))
    p.grad = _place(_grad(shape, dtype, view, span), view, dev)
    params = [p]
    for s, dt in companions:
        q = torch.nn.Parameter(torch.zeros(s, dtype=dt, device=dev))
        q.grad = torch.ones_like(q)
        params.append(q)
    opt = Gefen([("p%d" % i, q) for i, q in enumerate(params)], lr=1e-3)
    opt._gefen_codebook = _codebook(dev)
    for q in params:
        opt.state[q]["automatic_period"] = period if q is p else q.shape[1]
    opt.step()
    torch.cuda.synchronize()
    st = opt.state[p]
    return [p.detach().contiguous()] + [st[k].clone() for k in ("m_codebook", "m_magnitude", "v_row", "v_col")]


def _same(a, b):
    return all(torch.equal(x.contiguous().view(-1).view(torch.uint8), y.contiguous().view(-1).view(torch.uint8))
               for x, y in zip(a, b))


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dx%d-P%d-%s%s" % (
    c[0] + (c[1], str(c[2])[6:], "-view" if c[3] else "")))
def test_other_tensors_of_the_call(dev, case):
    alone = _step(dev, case, [])
    # 67M elements of the same launch; the same in another dtype; 1.1e9
    big = [((16384, 4096), case[2])]
    for others in (big, [((16384, 4096), F16)] + big, [((65536, 16384), case[2])]):
        assert _same(alone, _step(dev, case, others)), others


@pytest.mark.parametrize("case", [c for c in CASES if not c[3]], ids=lambda c: "%dx%d-P%d-%s" % (
    c[0] + (c[1], str(c[2])[6:])))
def test_scratch_and_entry_point(dev, case):
    """gefenx_factored_update with the required workspace and with more, and
    gefenx_factored_update_noalloc."""
    from gefen.kernels import _native
    from gefen.kernels import automatic_gefen_fused as fused
    (rows, cols), period, dtype, view, span = case
    lib, cb = _native.load(), _codebook(dev)
    qt = fused.quant_table(cb, dtype)
    need = int(lib.gefenx_workspace_bytes(_native.WS_FACTORED, rows, cols, rows * cols // period))
    outs = []
    for extra in (0, rows * cols // 4, None):
        g = _grad((rows, cols), dtype, view, span).to(dev)
        nb = rows * cols // period
        st = [torch.zeros_like(g), torch.zeros(rows * cols, dtype=torch.uint8, device=dev),
              torch.zeros(nb, device=dev), torch.zeros(rows, device=dev), torch.zeros(cols, device=dev)]
        args = [st[0].data_ptr(), g.data_ptr(), fused._dtype_code(dtype), rows, cols, cols, 1, cols, 1,
                *[t.data_ptr() for t in st[1:]], period, qt.data_ptr(), 0.9, 0.999, 1e-3, 1e-8, 1 / (1 - 0.999),
                1 / (1 - 0.9), 1.0, 0, 0, None, None]
        stream = torch.cuda.current_stream().cuda_stream
        if extra is None:
            rc = lib.gefenx_factored_update_noalloc(*args, stream)
        else:
            ws = torch.zeros(need + extra, dtype=torch.uint8, device=dev)
            rc = lib.gefenx_factored_update(*args, ws.data_ptr(), ws.numel(), stream)
        _native.check(rc, "factored update")
        torch.cuda.synchronize()
        outs.append(st)
    assert _same(outs[0], outs[1]) and _same(outs[0], outs[2])


def test_host_resident_chunks(dev, monkeypatch):
    """A host parameter is stepped with its chunk, a device parameter with the
    whole set."""
    from gefen import Gefen
    shape, period, dtype, view, span = CASES[0]
    outs = []
    for device in (torch.device("cpu"), dev):
        monkeypatch.setenv("GEFENX_HOST_STAGING_BYTES", str(8 << 20))
        params = []
        for s in (shape, (16384, 4096)):
            q = torch.nn.Parameter(torch.zeros(s, dtype=dtype, device=device))
            q.grad = (_grad(s, dtype, view, span) if s == shape else torch.ones(s, dtype=dtype)).to(device)
            params.append(q)
        opt = Gefen([("p%d" % i, q) for i, q in enumerate(params)], lr=1e-3)
        opt._gefen_codebook = _codebook(device)
        for q in params:
            opt.state[q]["automatic_period"] = q.shape[1]
        opt.step()
        torch.cuda.synchronize()
        st = opt.state[params[0]]
        outs.append([params[0].detach().cpu()] + [st[k].cpu() for k in ("m_codebook", "m_magnitude", "v_row", "v_col")])
    assert _same(outs[0], outs[1])
