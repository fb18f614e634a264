"""Sizes of the per-parameter workspace and of the call's scratch (host only)."""
from __future__ import annotations

import ctypes
import warnings

import pytest
import torch

from gefen.kernels import _native


@pytest.fixture(scope="module")
def lib():
    return _native.load()


@pytest.mark.parametrize("rows,cols", [(4096, 4096), (14336, 4096), (1024, 4096), (2048, 2048), (9728, 2560),
                                       (128256, 4096)])
def test_workspace_stays_small(lib, rows, cols):
    """What a parameter keeps between steps: with rows as blocks at most 0.14
    bytes per element (2048 x 2048: 32 shards of a block's 2048 elements are
    0.0625, its tiles' sums the rest), 0.05 over the Llama-3-8B set."""
    assert lib.gefenx_workspace_bytes(_native.WS_FACTORED, rows, cols, rows) <= 0.14 * rows * cols


def test_llama_layer_workspaces(lib):
    shapes = [(4096, 4096)] * 2 + [(1024, 4096)] * 2 + [(14336, 4096)] * 2 + [(4096, 14336)]
    total = sum(lib.gefenx_workspace_bytes(_native.WS_FACTORED, r, c, r) for r, c in shapes)
    assert total <= 0.055 * sum(r * c for r, c in shapes)


def _descs(specs):
    d = (_native.TensorDesc * len(specs))()
    for x, (rows, cols, dtype) in zip(d, specs):
        for f in ("p", "grad", "m_codebook", "m_magnitude", "v0", "v1", "workspace"):
            setattr(x, f, 4096)
        x.rows, x.cols, x.period, x.dtype, x.factored = rows, cols, cols, dtype, 1
        x.ps0 = x.gs0 = cols
        x.ps1 = x.gs1 = 1
    return d


def _extra(lib, specs):
    d = _descs(specs)
    n = len(specs)
    return lib.gefenx_multi_tensor_scratch_bytes_for(ctypes.addressof(d), n) - lib.gefenx_multi_tensor_scratch_bytes(n)


def test_scratch_follows_the_launches(lib):
    """A launch that would leave CUs idle gets scratch for finer sums, whatever
    launches of another dtype stand beside it; a launch of billions none."""
    f32, bf16 = _native.DT_F32, _native.DT_BF16
    one = _extra(lib, [(4096, 4096, f32)])
    assert one == 4096 * 4096 // 32 * 8
    large = [(128256, 4096, bf16)] * 4
    assert _extra(lib, large) == 0
    assert _extra(lib, large + [(4096, 4096, f32)]) == one
    assert _extra(lib, large + [(4096, 4096, bf16)]) == 0
    assert 0 < _extra(lib, [(14336, 4096, bf16)] * 6 + [(4096, 4096, bf16)] * 4) <= 64 << 20
    assert _extra(lib, [(64, 64, f32)] * 20) == 0


def test_workspace_memo_traces_without_a_warning(lib):
    """torch.compile of a step reaches the memo; a functools cache there made it
    warn that Dynamo ignores the cache."""
    from gefen import gefen
    key = (_native.WS_FACTORED, 64, 64, 64)
    gefen._workspace_bytes(*key)

    def f(x):
        return x + gefen._workspace_bytes(*key)

    torch._dynamo.reset()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        y = torch.compile(f, backend="eager")(torch.zeros(2))
    assert y[0].item() == lib.gefenx_workspace_bytes(*key)


@pytest.mark.parametrize("rows,cols", [(4096, 4096), (4096, 8), (8, 14336), (1, 4096), (65, 1000)])
def test_newton_schulz_batches_keep_their_budget(lib, rows, cols):
    """The matrices of one batch fit the budget with their padded buffers."""
    from gefen import GefenMuon
    from gefen.gefen_muon import NS_WORKSPACE_BUDGET
    opt = GefenMuon([("w", torch.nn.Parameter(torch.zeros(rows, cols)))], lr=1e-3)
    n = opt._ns_batch_limit(rows, cols, 2)
    assert n == 1 or lib.gefenx_ns_workspace_bytes(n, rows, cols) <= NS_WORKSPACE_BUDGET
    one = lib.gefenx_ns_workspace_bytes(1, rows, cols) + 2 * rows * cols  # and the matrix in the stack
    assert (n + 1) * one > NS_WORKSPACE_BUDGET
