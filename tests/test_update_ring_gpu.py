"""Circular decode on 64-byte granules of the state lines (MI355X): every
window offset of a granule, windows that reach the next granule and wrap at
the line's end, bursts of 1 to 8 tokens, channels and batches that do not fill
a wavefront, pools with padding entries; the state outside the window and the
pool's other rows stay as they were. A call large enough for granules to be
chosen over 16-byte chunks is checked once."""

from __future__ import annotations

import pytest
import torch

import causal_conv1d_amd as cc
from _util import DTYPE_IDS, DTYPES, assert_close
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(x, state, w, b, heads, idx, activation):
    sg = state.to(DEV)
    out = cc.causal_conv1d_update(x.to(DEV), sg, w.to(DEV), b.to(DEV), activation, cache_seqlens=heads.to(DEV),
                                  conv_state_indices=None if idx is None else idx.to(DEV))
    rs = state.clone()
    if idx is not None:  # an index past the pool acts as padding here (the oracle would write outside the pool)
        idx = torch.where(idx < state.shape[0], idx, -1)
    ref = O.causal_conv1d_update(x, rs, w, b, activation=activation, cache_seqlens=heads, conv_state_indices=idx)
    assert_close(out.cpu(), ref, x.dtype)
    assert torch.equal(sg.cpu(), rs)


# bursts that 16-byte chunks do not take (W-1 + tokens past a chunk) use granules at any size
@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("width,tokens", [(2, 8), (4, 7), (4, 8), (5, 5), (9, 3), (9, 8)])
@pytest.mark.parametrize("granules", [1, 2, 3])
@pytest.mark.parametrize("dim", [3, 64, 200])
def test_every_window_offset(dtype, width, tokens, granules, dim):
    S = granules * 64 // dtype.itemsize
    if width - 1 + tokens > 64 // dtype.itemsize:
        pytest.skip("the window is longer than a granule")
    B = S  # one batch entry per head position
    x, w, b = (torch.randn(*s).to(dtype) for s in ((B, dim, tokens), (dim, width), (dim,)))
    state = torch.randn(B, dim, S).to(dtype)
    heads = torch.arange(B, dtype=torch.int32) + torch.tensor([0, -S, S, 7 * S], dtype=torch.int32).repeat(B)[:B]
    _check(x, state, w, b, heads, None, "silu")


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("activation", [None, "silu"])
def test_pool_with_padding(dtype, activation):
    B, D, W, T = 13, 72, 4, 6
    S = 128 // dtype.itemsize
    x, w, b = (torch.randn(*s).to(dtype) for s in ((B, D, T), (D, W), (D,)))
    pool = torch.randn(20, D, S).to(dtype)
    idx = torch.randperm(20)[:B].to(torch.int32)
    idx[[0, 5]], idx[12] = -1, 20
    heads = torch.randint(0, S, (B,), dtype=torch.int32)
    _check(x, pool, w, b, heads, idx, activation)


def test_granules_chosen_by_size():
    """96 MiB of touched lines and more: one token and four, against the chunked kernel's bits."""
    B, D, S, W = 200, 4096, 64, 4
    for tokens in (1, 4):
        x, w, b = (torch.randn(*s, device=DEV).bfloat16() for s in ((B, D, tokens), (D, W), (D,)))
        big = torch.randn(B, D, S, device=DEV).bfloat16()
        small = big.clone()
        heads = torch.randint(0, S, (B,), dtype=torch.int32, device=DEV)
        out = cc.causal_conv1d_update(x, big, w, b, "silu", cache_seqlens=heads)
        parts = [cc.causal_conv1d_update(x[i:i + 50], small[i:i + 50], w, b, "silu", cache_seqlens=heads[i:i + 50])
                 for i in range(0, B, 50)]
        assert torch.equal(out, torch.cat(parts)) and torch.equal(big, small)
