"""Rows with a unit time stride on MI355X, wherever they lie: tensors that lie
unlike each other modulo 16 bytes (unaligned vectors), and rows of at most 32
vectors (several rows per wavefront). Each is held to the oracle on the same
inputs, at lengths around a vector, a wavefront's rows and a segment, with the
memory around every row left as it was."""

from __future__ import annotations

import ctypes

import pytest
import torch

import causal_conv1d_amd as cc
from causal_conv1d_amd import _lib, _native
from _util import DTYPE_IDS, DTYPES, assert_close, assert_reduction_close, make_inputs, scales, seq_pattern
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
GUARD = 7.0  # fills the memory around the rows


def _rows(t, lead, gap):
    """t on the GPU with `lead` elements before the first row and `gap` after each; the buffer too."""
    B, D, L = t.shape
    buf = torch.full((lead + B * D * (L + gap) + 64,), GUARD, dtype=t.dtype, device=DEV)
    v = buf[lead:lead + B * D * (L + gap)].view(B, D, L + gap)[..., :L]
    v.copy_(t)
    return v, buf


def _untouched(v, buf):
    """Everything of buf outside the view v still holds GUARD."""
    rest = buf.clone()
    torch.as_strided(rest, v.shape, v.stride(), v.storage_offset()).fill_(GUARD)
    return bool((rest == GUARD).all())


# (lead, gap) of x, out / dx, dout: every one different modulo the vector, or all tight
PLACES = {"tight": ((0, 0), (0, 0), (0, 0)), "unlike": ((1, 3), (2, 0), (5, 2)), "alike": ((1, 8), (1, 0), (1, 16))}


# lengths: below and around a vector, one row short of / over a power-of-two share of a wavefront,
# 31..33 vectors (the border to one row per wavefront), a segment's end
@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("place", list(PLACES))
@pytest.mark.parametrize("seqlen", [1, 3, 7, 8, 9, 17, 63, 124, 128, 129, 248, 255, 256, 257, 511, 1023, 2047, 2051])
@pytest.mark.parametrize("mode", ["plain", "seq_idx", "states"])
def test_rows_wherever_they_lie(dtype, place, seqlen, mode):
    B, D, W = 2, 37, 4  # 74 rows: no whole number of wavefronts
    activation = "silu" if seqlen % 2 else None
    x, w, b, _ = make_inputs(B, D, seqlen, W, dtype=dtype)
    dout = make_inputs(B, D, seqlen, W, dtype=dtype, seed=1)[0]
    seq = seq_pattern("repeat_ids", B, seqlen) if mode == "seq_idx" else None
    init = torch.randn(B, D, W - 1).to(dtype) if mode == "states" else None
    dfs = torch.randn(B, D, W - 1).to(dtype) if mode == "states" else None
    (px, po, pg) = PLACES[place]
    xg, xb = _rows(x, *px)
    og, ob = _rows(torch.zeros_like(x), *po)
    gg, gb = _rows(dout, *pg)
    dg, db_ = _rows(torch.zeros_like(x), *po)
    wg, bg = w.to(DEV), b.to(DEV)
    sg = None if seq is None else seq.to(DEV)
    ig = None if init is None else init.to(DEV)
    fg = None if init is None else torch.empty_like(ig)
    dw, dbias = torch.empty_like(wg), torch.empty_like(bg)
    di = None if init is None else torch.empty_like(ig)
    ops = torch.ops.causal_conv1d_amd
    ops._fwd_inplace(xg, wg, bg, sg, ig, og, activation is not None, fg)
    ops._bwd_typed_inplace(xg, wg, bg, gg, sg, ig, None if dfs is None else dfs.to(DEV), dg, dw, dbias, di,
                           activation is not None)
    torch.cuda.synchronize()
    for v, buf in ((xg, xb), (og, ob), (gg, gb), (dg, db_)):
        assert _untouched(v, buf)
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
    # the accumulating op on the same rows
    acc, bacc = torch.zeros(D, W, device=DEV), torch.zeros(D, device=DEV)
    d2 = torch.empty_like(xg)
    d3 = None if init is None else torch.empty_like(ig)
    ops._bwd_full_inplace(xg, wg, bg, gg, sg, ig, d2, acc, bacc, d3, activation is not None,
                          None if dfs is None else dfs.to(DEV))
    assert_close(d2.cpu(), rdx, dtype)  # (d2 is tight: with seq_idx its sums may associate another way than dg)
    assert_reduction_close(acc.cpu(), rdw.float(), dtype, scale=sw, name="dweight_acc")
    assert_reduction_close(bacc.cpu(), rdb.float(), dtype, scale=sb, name="dbias_acc")


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("width", [2, 3, 5, 9])
@pytest.mark.parametrize("seqlen", [1, 4, 13, 120])
def test_short_rows_widths(dtype, width, seqlen):
    if dtype == torch.float32 and width > 5:
        pytest.skip("fp32 widths above 5 are rejected by the API")
    B, D = 3, 50
    x, w, b, _ = make_inputs(B, D, seqlen, width, dtype=dtype)
    dout = make_inputs(B, D, seqlen, width, dtype=dtype, seed=1)[0]
    xg, wg, bg = (t.to(DEV).requires_grad_() for t in (x, w, b))
    out = cc.causal_conv1d_fn(xg, wg, bg, activation="silu")
    out.backward(dout.to(DEV))
    assert_close(out.detach().cpu(), O.causal_conv1d_fn(x, w, b, activation="silu"), dtype)
    rdx, rdw, rdb, _ = O.causal_conv1d_bwd(x, w, b, dout, activation="silu")
    assert_close(xg.grad.cpu(), rdx, dtype)
    sw, sb = scales(x, w, b, dout, activation="silu")
    assert_reduction_close(wg.grad.cpu(), rdw, dtype, scale=sw, name="dweight")
    assert_reduction_close(bg.grad.cpu(), rdb, dtype, scale=sb, name="dbias")


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("activation", [None, "silu"])
@pytest.mark.parametrize("seqlen", [5, 21, 64])
@pytest.mark.parametrize("mode", ["plain", "seq_idx"])
def test_nonfinite_rows_stay_with_their_row(dtype, activation, seqlen, mode):
    """A wavefront's rows share lanes' windows: inf and NaN at one row's ends reach no other row."""
    B, D, W = 2, 24, 4
    x, w, b, _ = make_inputs(B, D, seqlen, W, dtype=dtype)
    dout = make_inputs(B, D, seqlen, W, dtype=dtype, seed=1)[0]
    x[:, 6, 0], x[:, 6, -1] = float("nan"), float("inf")
    seq = seq_pattern("repeat_ids", B, seqlen) if mode == "seq_idx" else None
    xg, wg, bg = (t.to(DEV).requires_grad_() for t in (x, w, b))
    out = cc.causal_conv1d_fn(xg, wg, bg, seq_idx=None if seq is None else seq.to(DEV), activation=activation)
    out.backward(dout.to(DEV))
    ref = O.causal_conv1d_fn(x, w, b, seq_idx=seq, activation=activation)
    rdx, rdw, rdb, _ = O.causal_conv1d_bwd(x, w, b, dout, seq_idx=seq, activation=activation)
    keep = [c for c in range(D) if c != 6]
    for got, want in ((out.detach().cpu()[:, keep], ref[:, keep]), (xg.grad.cpu()[:, keep], rdx[:, keep]),
                      (wg.grad.cpu()[keep], rdw[keep]), (bg.grad.cpu()[keep], rdb[keep])):
        assert torch.isfinite(got).all() and torch.isfinite(want).all()
    assert_close(out.detach().cpu()[:, keep], ref[:, keep], dtype)
    assert_close(xg.grad.cpu()[:, keep], rdx[:, keep], dtype)
    assert torch.equal(torch.isfinite(out.detach().cpu()), torch.isfinite(ref))


@pytest.mark.parametrize("off", [0, 1])  # every tensor's first row, in elements past a 16-byte boundary
@pytest.mark.parametrize("seqlen", [3066, 3071, 3072, 5114, 5119, 5120])
def test_partial_sums_stay_in_the_workspace(seqlen, off):
    """Lengths whose vectors, counted from a row's first element and from the 16-byte boundary
    before it, are split into another number of segments: the floats behind the workspace
    stay as they were, and the sums are right."""
    B, D, W, dtype = 2, 48, 4, torch.bfloat16
    x, w, b, _ = make_inputs(B, D, seqlen, W, dtype=dtype)
    dout = make_inputs(B, D, seqlen, W, dtype=dtype, seed=1)[0]
    (xg, _), (gg, _), (dg, _) = (_rows(t, off, 0) for t in (x, dout, torch.zeros_like(x)))
    wg, bg = w.to(DEV), b.to(DEV)
    dw, db = torch.empty_like(wg), torch.empty_like(bg)
    p = _native._bwd_params(xg, wg, bg, gg, None, None, dg, None, True, None)
    lib = _lib.load()
    n = lib.cc1d_bwd_workspace_floats(ctypes.byref(p))
    ws = torch.full((2 * n,), GUARD, device=DEV)
    g = _lib.BwdGrads()
    g.dweight, g.dbias, g.workspace, g.workspace_floats = dw.data_ptr(), db.data_ptr(), ws.data_ptr(), n
    g.dweight_stride[:] = (W, 1)
    g.dbias_stride = 1
    assert lib.cc1d_bwd_typed(ctypes.byref(p), ctypes.byref(g), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert bool((ws[n:] == GUARD).all())
    rdx, rdw, rdb, _ = O.causal_conv1d_bwd(x, w, b, dout, activation="silu")
    assert_close(dg.cpu(), rdx, dtype)
    sw, sb = scales(x, w, b, dout, activation="silu")
    assert_reduction_close(dw.cpu(), rdw, dtype, scale=sw, name="dweight")
    assert_reduction_close(db.cpu(), rdb, dtype, scale=sb, name="dbias")


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("place", list(PLACES))
@pytest.mark.parametrize("activation", [None, "silu"])
@pytest.mark.parametrize("seqlen", [2, 21, 64, 261, 1021, 2051])
@pytest.mark.parametrize("where", ["row", "sequence"])
def test_nonfinite_dout_stays_with_the_taps_it_has(dtype, place, activation, seqlen, where):
    """dout of channel 6 is NaN at its row's first position, or at the first position of the row's
    second sequence: the reference adds no term there for the taps before (bwd_full_cpu/
    kernel.mojo:264-274), so only the channel's last tap and its bias are NaN. (Rows of more than
    32 vectors that lie alike take aligned vectors, which add a product with zero at a row's start:
    test_ragged_gpu.py's expected failures.)"""
    if where == "row" and place != "unlike" and seqlen > 64:
        pytest.skip("aligned vectors")
    B, D, W = 2, 12, 4
    x, w, b, _ = make_inputs(B, D, seqlen, W, dtype=dtype)
    dout = make_inputs(B, D, seqlen, W, dtype=dtype, seed=1)[0]
    seq = None
    if where == "sequence":
        seq = torch.zeros(B, seqlen, dtype=torch.int32)
        seq[:, seqlen // 2:] = 1
    dout[:, 6, 0 if seq is None else seqlen // 2] = float("nan")
    (px, po, pg) = PLACES[place]
    (xg, _), (gg, _), (dg, _) = _rows(x, *px), _rows(dout, *pg), _rows(torch.zeros_like(x), *po)
    wg, bg = w.to(DEV), b.to(DEV)
    dw, db = torch.empty_like(wg), torch.empty_like(bg)
    torch.ops.causal_conv1d_amd._bwd_typed_inplace(xg, wg, bg, gg, None if seq is None else seq.to(DEV), None, None, dg,
                                                   dw, db, None, activation is not None)
    rdx, rdw, rdb, _ = O.causal_conv1d_bwd(x, w, b, dout, seq_idx=seq, activation=activation)
    sw, sb = scales(x, w, b, torch.nan_to_num(dout), seq_idx=seq, activation=activation)
    assert int((~torch.isfinite(rdw.double())).sum()) == 1, "the case is what it says"
    for got, want, scale in ((dg, rdx, None), (dw, rdw, sw), (db, rdb, sb)):
        got, fin = got.cpu(), torch.isfinite(want.double())
        assert torch.equal(torch.isfinite(got.double()), fin)
        if scale is None:
            assert_close(got[fin], want[fin], dtype)
        else:
            assert_reduction_close(got[fin], want[fin], dtype, scale=scale[fin])
