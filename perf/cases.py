"""Performance cases of the causal conv1d framework.

Each case is one pass of what a program does with the public entry points:

* ``train``   -- ``causal_conv1d_fn`` forward and its autograd backward;
* ``prefill`` -- ``causal_conv1d_fn`` without gradients, returning the state
  that decoding goes on from: ``final_states``, or for packed sequences
  ``causal_conv1d_varlen_states`` of the same tokens;
* ``decode``  -- ``causal_conv1d_update`` with new tokens.

Layouts of x: ``rows`` is a contiguous (batch, dim, seqlen); ``half`` the
first half of the channels of a (batch, 2 * dim, seqlen) projection; ``last``
a (batch, seqlen, dim) buffer seen as (batch, dim, seqlen); ``part`` a time
slice [start, start + seqlen) of a longer (batch, dim, total) prompt, as in
chunked prefill.

Layouts of the decode state: ``line`` keeps each channel's state_len values
together (what ``final_states`` has), ``step`` keeps each step's dim values
together (what ``causal_conv1d_varlen_states`` returns), ``ring`` is a
circular buffer of lines addressed by ``cache_seqlens``.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

_PKG = str(Path(__file__).resolve().parent.parent / "causal-conv1d-mojo_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import causal_conv1d_amd as cc  # noqa: E402

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
LARGEST = 8 * 2048 * 16384 * 4  # bytes of x in the largest listed case


def _train(name, dtype, batch, dim, seqlen, layout, width=4, bias=True, silu=True, extra="none", seqs=1):
    return {"name": name, "op": "train", "dtype": dtype, "batch": batch, "dim": dim, "seqlen": seqlen,
            "width": width, "layout": layout, "bias": bias, "silu": silu, "extra": extra, "seqs": seqs}


def _prefill(name, dtype, batch, dim, seqlen, layout, width=4, bias=True, silu=True, extra="states", seqs=1,
             start=0, total=0):
    return {"name": name, "op": "prefill", "dtype": dtype, "batch": batch, "dim": dim, "seqlen": seqlen,
            "width": width, "layout": layout, "bias": bias, "silu": silu, "extra": extra, "seqs": seqs,
            "start": start, "total": total or start + seqlen}


def _decode(name, dtype, batch, dim, state, tokens=1, width=4, state_len=3, rows=0, padded=0, bias=True, silu=True):
    return {"name": name, "op": "decode", "dtype": dtype, "batch": batch, "dim": dim, "seqlen": tokens,
            "width": width, "layout": state, "bias": bias, "silu": silu, "state_len": state_len, "rows": rows,
            "padded": padded}


def listed():
    return [
        # one user's next token: nothing but latency
        _decode("decode one", "bf16", 1, 1536, "line"),
        # a serving batch whose sequences live at random rows of a state pool, some slots unused
        _decode("decode pool", "bf16", 256, 5120, "line", rows=512, padded=6),
        # a serving batch with circular states, four tokens a call
        _decode("decode ring", "bf16", 256, 5120, "ring", tokens=4, state_len=64),
        # decoding on the states that a packed prefill's state gather returned
        _decode("decode gathered", "bf16", 128, 4096, "step"),
        # a short prompt of any length
        _prefill("prefill short", "fp16", 1, 1536, 131, "half"),
        # one chunk of a long prompt, cut where the scheduler's token budget ends
        _prefill("prefill chunk", "bf16", 2, 4096, 1000, "part", start=1333, total=4099),
        # eight prompts packed into one sequence, and their states for decoding
        _prefill("prefill packed", "bf16", 1, 4096, 8192, "last", extra="packed", seqs=8),
        # a small layer's training step
        _train("train small", "bf16", 2, 768, 512, "half"),
        # a large layer's training step
        _train("train rows", "bf16", 4, 5120, 2048, "rows"),
        # packed documents of a batch that is not padded to a round length
        _train("train ragged", "fp16", 4, 5120, 2041, "rows", extra="packed", seqs=8),
        # a long sequence in channel-last memory, its state handed on from chunk to chunk
        _train("train last", "bf16", 1, 4096, 8192, "last", extra="states"),
        # long rows in 32 bits
        _train("train long", "fp32", 8, 2048, 16384, "rows", width=3, bias=False, silu=False),
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], even over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _dim(rng, low, high):
    """Channels: mostly a multiple of 64 or 8, as model sizes are, at times any number."""
    d = _spread(rng, low, high)
    unit = rng.choice((64, 64, 8, 1))
    return max(unit, d // unit * unit)


def draw(rng):
    op = rng.choice(("train", "train", "prefill", "decode"))
    dtype = rng.choice(("bf16", "bf16", "fp16", "fp32"))
    width = rng.choice((4, 4, 4, 4, 2, 3, 5, 5 if dtype == "fp32" else rng.randint(6, 9)))
    size = 4 if dtype == "fp32" else 2
    bias, silu = rng.random() < 0.8, rng.random() < 0.8
    if op == "decode":
        state = rng.choice(("line", "line", "ring", "step"))
        batch, dim = _spread(rng, 1, 512), _dim(rng, 64, 8192)
        tokens = rng.choice((1, 1, 1, rng.randint(2, 8)))
        state_len = width - 1
        if state == "ring":
            state_len = rng.choice((16, 32, 64, 128))
        elif rng.random() < 0.2:
            state_len += rng.randint(1, 4)
        rows, padded = 0, 0
        if state != "ring" and rng.random() < 0.5:
            rows, padded = batch + _spread(rng, 1, 512), rng.choice((0, 0, batch // 8))
        c = _decode("", dtype, batch, dim, state, tokens, width, state_len, rows, padded, bias, silu)
    else:
        batch, dim, seqlen = _spread(rng, 1, 16), _dim(rng, 64, 8192), _spread(rng, 16, 16384)
        if rng.random() < 0.5:
            seqlen = max(1, seqlen // 64) * 64
        most = LARGEST // (2 if op == "prefill" else 1)
        while batch * dim * seqlen * size > most:
            batch, seqlen = (batch + 1) // 2, seqlen if batch > 1 else seqlen // 2
        extra = rng.choice(("none", "packed", "states"))
        seqs = max(1, min(seqlen // 8, rng.randint(1, 16))) if extra == "packed" else 1
        layout = rng.choice(("rows", "half", "last"))
        if op == "train":
            c = _train("", dtype, batch, dim, seqlen, layout, width, bias, silu, extra, seqs)
        else:
            if extra == "states":
                layout = rng.choice((layout, layout, "part"))
            start = rng.randint(0, 2048) if layout == "part" else 0
            total = start + seqlen + (rng.randint(0, 2048) if layout == "part" else 0)
            while batch * dim * total * size > LARGEST:
                start, total = start // 2, start // 2 + seqlen
            c = _prefill("", dtype, batch, dim, seqlen, layout, width, bias, silu, extra, seqs, start, total)
    del c["name"]
    return c


def _activations(gen, dtype, *shape):
    return torch.randn(*shape, generator=gen, device=DEVICE, dtype=torch.float32).to(dtype)


def _parameters(c, gen, dtype):
    """Weight and bias as a depthwise conv layer initialises them."""
    bound = 1.0 / math.sqrt(c["width"])
    weight = (torch.rand(c["dim"], c["width"], generator=gen, device=DEVICE) * 2 - 1) * bound
    bias = (torch.rand(c["dim"], generator=gen, device=DEVICE) * 2 - 1) * bound
    return weight.to(dtype), bias.to(dtype) if c["bias"] else None


def _input(c, gen, dtype):
    B, D, L = c["batch"], c["dim"], c["seqlen"]
    if c["layout"] == "last":
        return _activations(gen, dtype, B, L, D).transpose(1, 2)
    if c["layout"] == "half":
        return _activations(gen, dtype, B, 2 * D, L)[:, :D]
    if c["layout"] == "part":
        return _activations(gen, dtype, B, D, c["total"])[..., c["start"]:c["start"] + L]
    return _activations(gen, dtype, B, D, L)


def _ids(c, seed):
    """Sequence ids (batch, seqlen) of seqs sequences of random lengths a row, and each row's boundaries."""
    cpu = torch.Generator().manual_seed(seed)
    B, L, n = c["batch"], c["seqlen"], c["seqs"]
    cuts = torch.stack([torch.randperm(L - 1, generator=cpu)[:n - 1].sort().values + 1 if n > 1
                        else torch.empty(0, dtype=torch.int64) for _ in range(B)])
    marks = torch.zeros(B, L, dtype=torch.int32)
    marks.scatter_(1, cuts, 1)
    bounds = F.pad(F.pad(cuts, (1, 0)), (0, 1), value=L)
    return marks.cumsum(1, dtype=torch.int32).to(DEVICE), bounds


def prepare(case, seed):
    c = case
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = DTYPES[c["dtype"]]
    B, D, L, W = c["batch"], c["dim"], c["seqlen"], c["width"]
    weight, bias = _parameters(c, gen, dtype)
    s = {"case": c, "weight": weight, "bias": bias, "activation": "silu" if c["silu"] else None}
    if c["op"] == "decode":
        shape = (c["rows"] or B, D, c["state_len"])
        if c["layout"] == "step":
            s["state"] = _activations(gen, dtype, shape[0], shape[2], shape[1]).transpose(1, 2)
        else:
            s["state"] = _activations(gen, dtype, *shape)
        s["x"] = _activations(gen, dtype, B, D) if L == 1 else _activations(gen, dtype, B, D, L)
        cpu = torch.Generator().manual_seed(seed)
        s["indices"] = s["heads"] = None
        if c["rows"]:
            indices = torch.randperm(c["rows"], generator=cpu)[:B].to(torch.int32)
            if c["padded"]:
                indices[-c["padded"]:] = -1  # a captured batch size is filled up with unused slots
            s["indices"] = indices.to(DEVICE)
        if c["layout"] == "ring":
            s["heads"] = torch.randint(0, c["state_len"], (B,), generator=cpu, dtype=torch.int32).to(DEVICE)
        return s
    s["x"] = _input(c, gen, dtype)
    s["ids"] = s["bounds"] = s["initial"] = None
    if c["extra"] == "packed":
        s["ids"], bounds = _ids(c, seed)
        s["bounds"] = (bounds[0].to(torch.int32)).to(DEVICE) if B == 1 else None
    if c["extra"] == "states":
        s["initial"] = _activations(gen, dtype, B, D, W - 1)
    if c["op"] == "train":
        s["dout"] = torch.empty_like(s["x"]).normal_(generator=gen)
        s["dfinal"] = _activations(gen, dtype, B, D, W - 1) if c["extra"] == "states" else None
        for k in ("x", "weight", "bias", "initial"):
            if s[k] is not None:
                s[k].requires_grad_()
    return s


def run(state):
    s = state
    c = s["case"]
    if c["op"] == "decode":
        out = cc.causal_conv1d_update(s["x"], s["state"], s["weight"], s["bias"], s["activation"],
                                      cache_seqlens=s["heads"], conv_state_indices=s["indices"])
        return {"out": out, "state": s["state"]}
    states = c["extra"] == "states"
    if c["op"] == "prefill":
        with torch.no_grad():
            out = cc.causal_conv1d_fn(s["x"], s["weight"], s["bias"], seq_idx=s["ids"], initial_states=s["initial"],
                                      return_final_states=states, activation=s["activation"])
            if states:
                return {"out": out[0], "final": out[1]}
            if s["bounds"] is None or c["layout"] != "last":
                return {"out": out}
            return {"out": out, "states": cc.causal_conv1d_varlen_states(s["x"][0].t(), s["bounds"], c["width"] - 1)}
    out = cc.causal_conv1d_fn(s["x"], s["weight"], s["bias"], seq_idx=s["ids"], initial_states=s["initial"],
                              return_final_states=states, activation=s["activation"])
    wanted = {k: s[k] for k in ("x", "weight", "bias", "initial") if s[k] is not None}
    if states:
        out, final = out
        grads = torch.autograd.grad((out, final), tuple(wanted.values()), (s["dout"], s["dfinal"]))
    else:
        grads = torch.autograd.grad(out, tuple(wanted.values()), s["dout"])
    got = {"out": out}
    if states:
        got["final"] = final
    got.update({"d" + k: g for k, g in zip(wanted, grads)})
    return got


def work(case):
    c = case
    size = 4 if c["dtype"] == "fp32" else 2
    B, D, L, W = c["batch"], c["dim"], c["seqlen"], c["width"]
    n, H = B * D * L, c["width"] - 1
    params = D * (W + (1 if c["bias"] else 0)) * size
    forward = (2 * W + (4 if c["silu"] else 0)) * n
    if c["op"] == "decode":
        live = (B - c["padded"]) * D
        S = c["state_len"]
        if c["layout"] == "ring":  # the window is read, the new tokens are written
            state = live * (H + L)
        else:  # what stays is read and moved, or read as history; the whole line is written
            state = live * (max(S - L, H) + S)
        index = 4 * B * ((1 if c["rows"] else 0) + (1 if c["layout"] == "ring" else 0))
        return {"bytes": (2 * n + state) * size + params + index, "flops": forward}
    ids = 4 * B * L if c["extra"] == "packed" else 0
    states = B * D * H * size if c["extra"] == "states" else 0
    moved = 2 * n * size + params + ids + 2 * states
    if c["op"] == "prefill":
        if c["extra"] == "packed" and B == 1 and c["layout"] == "last":
            moved += c["seqs"] * D * H * size
        return {"bytes": moved, "flops": forward}
    # backward: x, dout and the parameters in, dx and their gradients out
    moved += 3 * n * size + 2 * params + ids + 3 * states
    return {"bytes": moved, "flops": forward + (6 * W + (9 if c["silu"] else 0)) * n}


def tolerance(case):
    # about four times the largest distance from exact() seen: 1.7e-3 and 2.1e-4 are the rounding
    # of one result to bf16 and fp16; in 32 bits 1.4e-7 (the weight gradient's sums, 131072 terms),
    # with room for SiLU's exponential and reciprocal and for sums in another order
    return {"rel": {"bf16": 7e-3, "fp16": 9e-4, "fp32": 1e-6}[case["dtype"]]}


def _taps(x, initial, W):
    return torch.cat([torch.zeros(*x.shape[:2], W - 1, dtype=x.dtype, device=x.device) if initial is None else initial,
                      x], -1)


def _exact_decode(c, s):
    W, H, L, S = c["width"], c["width"] - 1, c["seqlen"], c["state_len"]
    x = s["x"].double().reshape(c["batch"], c["dim"], L)
    rows = torch.arange(c["batch"], device=DEVICE) if s["indices"] is None else s["indices"].long()
    live = rows >= 0
    state = s["state"].double()
    lines = state[rows.clamp(min=0)]
    if s["heads"] is None:
        history = lines[..., S - H:]
        lines = torch.cat([lines, x], -1)[..., L:]
    else:
        head = s["heads"].long()[:, None]
        at = ((head - H + torch.arange(H, device=DEVICE)) % S)[:, None].expand(-1, c["dim"], -1)
        history = lines.gather(-1, at)
        lines.scatter_(-1, ((head + torch.arange(L, device=DEVICE)) % S)[:, None].expand(-1, c["dim"], -1), x)
    full = torch.cat([history, x], -1)
    out = sum(s["weight"].double()[:, k, None] * full[..., k:k + L] for k in range(W))
    if s["bias"] is not None:
        out = out + s["bias"].double()[:, None]
    if c["silu"]:
        out = out * torch.sigmoid(out)
    out[~live] = 0.0
    state[rows[live]] = lines[live]
    return {"out": out.reshape(s["x"].shape), "state": state}


def _exact_channels(c, s, at):
    """Results of the channels `at` (a slice), as run() names them."""
    W, H, L = c["width"], c["width"] - 1, c["seqlen"]
    x = s["x"].detach()[:, at].double()
    w = s["weight"].detach()[at].double()
    initial = None if s["initial"] is None else s["initial"].detach()[:, at].double()
    full = _taps(x, initial, W)
    kept = None
    if s["ids"] is not None:
        before = F.pad(s["ids"], (H, 0), value=-1)
        kept = [(before[:, k:k + L] == s["ids"])[:, None] for k in range(W)]

    def tap(k, of):
        return of if kept is None else torch.where(kept[k], of, 0.0)

    pre = sum(w[:, k, None] * tap(k, full[..., k:k + L]) for k in range(W))
    if s["bias"] is not None:
        pre += s["bias"].detach()[at].double()[:, None]
    sig = torch.sigmoid(pre) if c["silu"] else None
    got = {"out": pre * sig if c["silu"] else pre}
    if c["extra"] == "states":
        got["final"] = F.pad(x, (H, 0))[..., L:]
    if c["op"] != "train":
        return got
    d = s["dout"][:, at].double()
    if c["silu"]:
        d = d * sig * (1.0 + pre * (1.0 - sig))
    dfull = torch.zeros_like(full)
    dw = torch.empty_like(w)
    for k in range(W):
        dw[:, k] = (d * tap(k, full[..., k:k + L])).sum((0, 2))
        dfull[..., k:k + L] += w[:, k, None] * tap(k, d)
    got["dx"] = dfull[..., H:]
    if s["dfinal"] is not None:
        m = min(H, L)
        got["dx"][..., L - m:] += s["dfinal"][:, at].double()[..., H - m:]
    got["dweight"] = dw
    if s["bias"] is not None:
        got["dbias"] = d.sum((0, 2))
    if initial is not None:
        got["dinitial"] = dfull[..., :H]
    return got


def exact(case, seed):
    c = case
    s = prepare(c, seed)
    if c["op"] == "decode":
        return _exact_decode(c, s)
    B, D, L, W = c["batch"], c["dim"], c["seqlen"], c["width"]
    step = max(1, min(D, (1 << 26) // (B * (L + W))))
    parts = [_exact_channels(c, s, slice(i, i + step)) for i in range(0, D, step)]
    got = {k: torch.cat([p[k] for p in parts], 0 if k in ("dweight", "dbias") else 1) for k in parts[0]}
    if c["op"] == "prefill" and s["bounds"] is not None and c["layout"] == "last":
        ends = s["bounds"].tolist()
        states = torch.zeros(c["seqs"], D, W - 1, dtype=torch.float64, device=DEVICE)
        for i, (a, b) in enumerate(zip(ends, ends[1:])):
            n = min(W - 1, b - a)
            if n:
                states[i, :, W - 1 - n:] = s["x"][0, :, b - n:b].double()
        got["states"] = states
    return got
