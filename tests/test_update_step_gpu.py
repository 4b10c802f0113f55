"""Single-token linear decode on MI355X with states that are not lines of W-1
values: a step's channels together (as causal_conv1d_varlen_states returns
them), and lines or steps with room for more than W-1 values. The state moves
bit for bit; entries that are padding, and the pool's other rows, stay."""

from __future__ import annotations

import pytest
import torch

import causal_conv1d_amd as cc
from _util import DTYPE_IDS, DTYPES, assert_close
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("width,extra", [(2, 0), (2, 1), (3, 1), (4, 0), (4, 1), (4, 3), (5, 1), (5, 2), (9, 0), (9, 1)])
@pytest.mark.parametrize("layout", ["line", "step", "step slice"])
@pytest.mark.parametrize("batch,dim", [(1, 2), (5, 64), (2, 136), (3, 130), (4, 33), (2, 1032)])
@pytest.mark.parametrize("pool", [False, True])
def test_states(dtype, width, extra, layout, batch, dim, pool):
    S = width - 1 + extra
    x, w, b = (torch.randn(*s).to(dtype) for s in ((batch, dim), (dim, width), (dim,)))
    rows = batch + 3 if pool else batch
    state = torch.randn(rows, dim, S).to(dtype)
    idx = None
    if pool:
        idx = torch.randperm(rows)[:batch].to(torch.int32)
        if batch > 2:
            idx[1] = -1
    if layout == "line":
        sg = state.to(DEV)
    else:
        pad = 6 if layout == "step slice" else 0
        sg = torch.zeros(rows, S, dim + pad, dtype=dtype, device=DEV)[..., pad // 3:pad // 3 + dim].transpose(1, 2)
        sg.copy_(state)
    out = cc.causal_conv1d_update(x.to(DEV), sg, w.to(DEV), None if extra == 3 else b.to(DEV), "silu" if width % 2 else None,
                                  conv_state_indices=None if idx is None else idx.to(DEV))
    ref = O.causal_conv1d_update(x, state, w, None if extra == 3 else b, activation="silu" if width % 2 else None,
                                 conv_state_indices=idx)
    assert_close(out.cpu(), ref, dtype)
    assert torch.equal(sg.cpu(), state)
