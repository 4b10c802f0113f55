"""Channel-last tensors off the dword grid on MI355X: odd numbers of 16-bit
channels (the last lane shares a channel with the one before), channel slices
that start at an odd channel of a wider buffer, row strides that alternate the
alignment; with the channels around the slice left as they were."""

from __future__ import annotations

import pytest
import torch

from _util import DTYPE_IDS, DTYPES, assert_close, assert_reduction_close, make_inputs, scales, seq_pattern
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
GUARD = 7.0


def _slice(t, lead, gap):
    """t (B, D, L) on the GPU as channels [lead, lead + D) of a channel-last buffer of lead + D + gap channels."""
    B, D, L = t.shape
    buf = torch.full((B, L, lead + D + gap), GUARD, dtype=t.dtype, device=DEV)
    v = buf[..., lead:lead + D].transpose(1, 2)
    v.copy_(t)
    return v, buf


# (1, .): fewer channels than a lane holds; 129, 257: one channel past a wavefront's; 255: one short
@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("dim,lead,gap", [(1, 0, 0), (2, 1, 0), (3, 0, 0), (64, 1, 2), (127, 0, 0), (129, 3, 1), (255, 0, 0),
                                          (257, 0, 1)])
@pytest.mark.parametrize("seqlen", [2, 37, 260])
@pytest.mark.parametrize("mode", ["plain", "seq_idx", "states"])
def test_channels_off_the_dword_grid(dtype, dim, lead, gap, seqlen, mode):
    B, W = 2, 4
    activation = "silu" if dim % 2 else None
    x, w, b, _ = make_inputs(B, dim, seqlen, W, dtype=dtype)
    dout = make_inputs(B, dim, seqlen, W, dtype=dtype, seed=1)[0]
    seq = seq_pattern("repeat_ids", B, seqlen) if mode == "seq_idx" else None
    init = torch.randn(B, dim, W - 1).to(dtype) if mode == "states" else None
    dfs = torch.randn(B, dim, W - 1).to(dtype) if mode == "states" else None
    xg, xb = _slice(x, lead, gap)
    og, ob = _slice(torch.zeros_like(x), lead + 1, gap)
    gg, _ = _slice(dout, lead, gap + 1)
    dg, db_ = _slice(torch.zeros_like(x), lead, 0)
    wg, bg = w.to(DEV), b.to(DEV)
    sg, ig, dfg = (None if t is None else t.to(DEV) for t in (seq, init, dfs))
    fg = None if init is None else torch.empty_like(ig)
    dw, dbias, di = torch.empty_like(wg), torch.empty_like(bg), None if init is None else torch.empty_like(ig)
    ops = torch.ops.causal_conv1d_amd
    ops._fwd_inplace(xg, wg, bg, sg, ig, og, activation is not None, fg)
    ops._bwd_typed_inplace(xg, wg, bg, gg, sg, ig, dfg, dg, dw, dbias, di, activation is not None)
    for v, buf in ((og, ob), (dg, db_)):
        rest = buf.clone()
        torch.as_strided(rest, v.shape, v.stride(), v.storage_offset()).fill_(GUARD)
        assert bool((rest == GUARD).all())
    ref = O.causal_conv1d_fn(x, w, b, seq_idx=seq, initial_states=init, activation=activation,
                             return_final_states=init is not None)
    if init is not None:
        ref, rfs = ref
        assert torch.equal(fg.cpu(), rfs)
    assert_close(og.cpu(), ref, dtype)
    rdx, rdw, rdb, rdi = O.causal_conv1d_bwd(x, w, b, dout, seq_idx=seq, initial_states=init, dfinal_states=dfs,
                                             activation=activation)
    assert_close(dg.cpu(), rdx, dtype)
    sw, sb = scales(x, w, b, dout, seq_idx=seq, init=init, activation=activation)
    assert_reduction_close(dw.cpu(), rdw, dtype, scale=sw, name="dweight")
    assert_reduction_close(dbias.cpu(), rdb, dtype, scale=sb, name="dbias")
    if init is not None:
        assert_close(di.cpu(), rdi, dtype)
    acc, bacc = torch.zeros(dim, W, device=DEV), torch.zeros(dim, device=DEV)
    ops._bwd_full_inplace(xg, wg, bg, gg, sg, ig, dg, acc, bacc, di, activation is not None, dfg)
    assert_reduction_close(acc.cpu(), rdw.float(), dtype, scale=sw, name="dweight_acc")
    assert_reduction_close(bacc.cpu(), rdb.float(), dtype, scale=sb, name="dbias_acc")
