"""The native host path on MI355X: an ordinary call runs there, with the bits
and layouts of the Python path (the ops and the autograd Function), and every
call that something observes or transforms goes through the ops as before."""

from __future__ import annotations

import threading

import pytest
import torch
import torch.utils.checkpoint
from functorch.compile import make_boxed_func
from torch._dynamo.backends.common import aot_autograd
from torch.utils._python_dispatch import TorchDispatchMode

import causal_conv1d_amd as cc
from causal_conv1d_amd import _fn, _host

pytestmark = pytest.mark.gpu
DEV = "cuda"
B, D, L, W = 2, 24, 75, 4


def _args(mode, dtype=torch.bfloat16, grad=True, layout="rows"):
    torch.manual_seed(3)
    x = torch.randn(B, D, L, device=DEV).to(dtype)
    if layout == "last":
        x = x.transpose(1, 2).contiguous().transpose(1, 2)
    kw = dict(weight=torch.randn(D, W, device=DEV).to(dtype), bias=torch.randn(D, device=DEV).to(dtype), activation="silu")
    if mode == "seq":
        kw["seq_idx"] = (torch.arange(L, device=DEV, dtype=torch.int32) // 20).expand(B, L).contiguous()
    if mode == "states":
        kw.update(initial_states=torch.randn(B, D, W - 1, device=DEV).to(dtype), return_final_states=True)
    if mode == "nobias":
        kw.update(bias=None, activation=None)
    if grad:
        for t in (x, kw["weight"], kw["bias"], kw.get("initial_states")):
            if t is not None:
                t.requires_grad_()
    return x, kw


def _run(x, kw, dout, dfinal):
    r = cc.causal_conv1d_fn(x, **kw)
    out, final = r if isinstance(r, tuple) else (r, None)
    ins = [t for t in (x, kw["weight"], kw["bias"], kw.get("initial_states")) if t is not None]
    outs, douts = ([out, final], [dout, dfinal]) if final is not None else ([out], [dout])
    return [out, *([final] if final is not None else []), *torch.autograd.grad(outs, ins, douts)]


@pytest.fixture
def python_path(monkeypatch):
    """Turns the native path off inside the returned context."""
    def off():
        monkeypatch.setattr(_host, "native", lambda: type("Off", (), {
            n: staticmethod(lambda *a: NotImplemented) for n in ("fn", "update", "varlen_states")}))
    yield off
    monkeypatch.undo()


@pytest.mark.parametrize("mode", ["plain", "seq", "states", "nobias"])
@pytest.mark.parametrize("layout", ["rows", "last"])
@pytest.mark.parametrize("dout", ["like", "rows", "expanded"])
def test_same_bits_and_layouts(mode, layout, dout, python_path):
    x, kw = _args(mode, layout=layout)
    g = {"like": torch.randn_like(x), "rows": torch.randn(B, D, L, device=DEV).to(x.dtype),
         "expanded": torch.ones((), device=DEV, dtype=x.dtype).expand(B, D, L)}[dout]
    df = torch.randn(B, D, W - 1, device=DEV).to(x.dtype)
    got = _run(x, kw, g, df)
    python_path()
    want = _run(x, kw, g, df)
    for a, b in zip(got, want, strict=True):
        assert torch.equal(a, b) and a.stride() == b.stride() and a.dtype == b.dtype


def test_ordinary_calls_run_natively(monkeypatch):
    def never(*a, **k):
        raise AssertionError("the Python path ran")

    monkeypatch.setattr(_fn._CausalConv1dFn, "apply", never)
    for mode in ("plain", "seq", "states"):
        x, kw = _args(mode)
        r = cc.causal_conv1d_fn(x, **kw)
        (r[0] if isinstance(r, tuple) else r).float().sum().backward()
        assert x.grad is not None
        with torch.inference_mode():
            cc.causal_conv1d_fn(x.detach(), **{**kw, "bias": torch.nn.Parameter(kw["bias"].detach())})


@pytest.mark.parametrize("which", ["final only", "out only"])
def test_undefined_grads(which, python_path):
    x, kw = _args("states")
    def go():
        out, final = cc.causal_conv1d_fn(x, **kw)
        return torch.autograd.grad((final if which == "final only" else out).float().square().sum(), [x, kw["weight"]])
    got = go()
    python_path()
    for a, b in zip(got, go(), strict=True):
        assert torch.equal(a, b)


def test_dispatch_modes_see_the_ops():
    seen = []

    class Log(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    x, kw = _args("plain")
    with Log():
        cc.causal_conv1d_fn(x, **kw)
    assert any("_fwd_inplace" in s for s in seen)
    out = cc.causal_conv1d_fn(x, **kw)  # a native node, differentiated under the mode
    seen.clear()
    with Log():
        out.sum().backward()
    assert any("_bwd_typed_inplace" in s for s in seen)


def test_saved_tensor_hooks_and_versions():
    x, kw = _args("plain")
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(tuple(t.shape)) or t.cpu(), lambda t: t.to(DEV)):
        out = cc.causal_conv1d_fn(x, **kw)
    assert (B, D, L) in packed and (D, W) in packed
    got = torch.autograd.grad(out.sum(), x)[0]
    assert torch.equal(got, torch.autograd.grad(cc.causal_conv1d_fn(x, **kw).sum(), x)[0])
    out = cc.causal_conv1d_fn(x, **kw)
    with torch.no_grad():
        kw["weight"].mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


class _Sub(torch.Tensor):
    pass


def _outcome(f):
    try:
        r = f()
        return [t.detach() for t in (r if isinstance(r, (tuple, list)) else [r])]
    except Exception as e:  # noqa: BLE001 -- whatever the Python path does
        return type(e).__name__


@pytest.mark.parametrize("what", ["double backward", "create_graph", "forward-mode", "vmap", "func.grad", "subclass",
                                  "function mode", "final_states_out", "strided seq", "float heads"])
def test_everything_else_as_the_python_path(what, python_path):
    def go():
        x, kw = _args("plain")
        w, b = kw["weight"], kw["bias"]
        f = lambda t: cc.causal_conv1d_fn(t, w, b, activation="silu")  # noqa: E731
        if what == "double backward":
            g = torch.autograd.grad(f(x).float().square().sum(), x, create_graph=True)[0]
            return torch.autograd.grad(g.float().sum(), x)
        if what == "create_graph":
            return torch.autograd.grad(f(x).float().square().sum(), x, create_graph=True)
        if what == "forward-mode":
            with torch.autograd.forward_ad.dual_level():
                return f(torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x)))
        if what == "vmap":
            return torch.func.vmap(f)(x.detach()[None])
        if what == "func.grad":
            return torch.func.grad(lambda t: f(t).float().sum())(x.detach())
        if what == "subclass":
            return f(x.detach().as_subclass(_Sub))
        if what == "function mode":
            class Mode(torch.overrides.TorchFunctionMode):
                def __torch_function__(self, func, types, args=(), kwargs=None):
                    return func(*args, **(kwargs or {}))
            with Mode():
                return f(x)
        if what == "final_states_out":
            fs = torch.empty(B, D, W - 1, device=DEV, dtype=x.dtype)
            out, got = cc.causal_conv1d_fn(x, w, b, return_final_states=True, final_states_out=fs)
            assert got.data_ptr() == fs.data_ptr()
            return out, got
        if what == "strided seq":
            seq = torch.zeros(B, 2 * L, device=DEV, dtype=torch.int32)[:, ::2]
            return cc.causal_conv1d_fn(x, w, b, seq_idx=seq)
        return cc.causal_conv1d_update(x[..., 0].detach(), torch.zeros(B, D, 8, device=DEV, dtype=x.dtype), w, b,
                                       cache_seqlens=torch.zeros(B, device=DEV))
    got = _outcome(go)
    python_path()
    want = _outcome(go)
    if isinstance(want, str):
        assert got == want
    else:
        assert all(torch.equal(a, b) and type(a) is type(b) for a, b in zip(got, want, strict=True))


def test_update_and_states_same_bits(python_path):
    torch.manual_seed(5)
    x, w, b = (torch.randn(*s, device=DEV).half() for s in ((7, 48), (48, 4), (48,)))
    pool = torch.randn(9, 48, 3, device=DEV).half()
    idx = torch.tensor([3, -1, 0, 8, 9, 1, 2], dtype=torch.int32, device=DEV)
    cu = torch.tensor([0, 2, 2, 30], dtype=torch.int32, device=DEV)
    tok = torch.randn(31, 48, device=DEV).half()

    def go():
        s = pool.clone()
        out = cc.causal_conv1d_update(x, s, w, b, "silu", conv_state_indices=idx)
        ring = pool.repeat(1, 1, 3)[:7].contiguous()
        out3 = cc.causal_conv1d_update(x[..., None].expand(-1, -1, 2), ring, w, cache_seqlens=idx.clamp(min=0))
        return out, s, out3, ring, cc.causal_conv1d_varlen_states(tok, cu, 3)
    got = go()
    python_path()
    for a, c in zip(got, go(), strict=True):
        assert torch.equal(a, c) and a.stride() == c.stride()


def test_errors_as_before():
    x, kw = _args("plain")
    with pytest.raises(NotImplementedError, match="width must be in"):
        cc.causal_conv1d_fn(x, torch.randn(D, 10, device=DEV).to(x.dtype))
    with pytest.raises(ValueError, match="expected"):
        cc.causal_conv1d_fn(x, kw["weight"][:3])
    with pytest.raises(NotImplementedError, match="same device"):
        cc.causal_conv1d_fn(x, kw["weight"].cpu())
    with pytest.raises(ValueError, match="must be >="):
        cc.causal_conv1d_update(x[..., 0], torch.zeros(B, D, 2, device=DEV, dtype=x.dtype), kw["weight"])


def _step(x, kw, dout):
    """Fresh leaves, one training step: (out, dx, dweight, dbias)."""
    xs = x.detach().clone().requires_grad_()
    w, b = (kw[k].detach().clone().requires_grad_() for k in ("weight", "bias"))
    out = cc.causal_conv1d_fn(xs, w, b, activation="silu")
    return [out.detach(), *torch.autograd.grad(out, [xs, w, b], dout)]


def test_threads_each_on_a_stream_of_its_own():
    """The lock is given up while a call allocates and launches: calls of several threads interleave."""
    x, kw = _args("plain")
    douts = [torch.randn_like(x).detach() for _ in range(4)]
    want = [_step(x, kw, g) for g in douts]
    got, errors = {}, []
    torch.cuda.synchronize()

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                got[i] = [_step(x, kw, douts[i]) for _ in range(20)]
                torch.cuda.current_stream().synchronize()
        except BaseException as e:  # noqa: BLE001 -- reported below
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and len(got) == 4
    for i, runs in got.items():
        assert all(torch.equal(a, b) for run in runs for a, b in zip(run, want[i], strict=True))


def test_calls_follow_the_current_stream():
    """Inputs made late on a side stream: forward there, backward from outside the block."""
    x, kw = _args("plain")
    dout = torch.randn_like(x).detach()
    want = _step(x, kw, dout)
    state = torch.randn(B, D, W - 1, device=DEV).to(x.dtype)
    tok = x.detach()[..., 0].contiguous()
    ref_state = state.clone()
    ref_tok = cc.causal_conv1d_update(tok, ref_state, kw["weight"].detach())
    big = torch.randn(4096, 4096, device=DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        late = torch.zeros_like(x.detach())
        for _ in range(8):
            big = big @ big * 1e-3  # the inputs arrive after this
        late.copy_(x.detach())
        late.requires_grad_()
        w, b = (kw[k].detach().clone().requires_grad_() for k in ("weight", "bias"))
        out = cc.causal_conv1d_fn(late, w, b, activation="silu")
        own = state.clone()
        step = cc.causal_conv1d_update(late.detach()[..., 0].contiguous(), own, w.detach())
    torch.cuda.current_stream().wait_stream(side)
    grads = torch.autograd.grad(out, [late, w, b], dout)
    torch.cuda.synchronize()
    for a, c in zip([out.detach(), *grads, step, own], [*want, ref_tok, ref_state], strict=True):
        assert torch.equal(a, c)


@pytest.mark.parametrize("reentrant", [True, False])
def test_activation_checkpointing(reentrant):
    x, kw = _args("plain")
    dout = torch.randn_like(x).detach()
    want = _step(x, kw, dout)
    xs = x.detach().clone().requires_grad_()
    w, b = (kw[k].detach().clone().requires_grad_() for k in ("weight", "bias"))

    def f(t):
        return cc.causal_conv1d_fn(t, w, b, activation="silu")

    out = torch.utils.checkpoint.checkpoint(f, xs, use_reentrant=reentrant)
    out.backward(dout)
    for a, c in zip([out.detach(), xs.grad, w.grad, b.grad], want, strict=True):
        assert torch.equal(a, c)


@pytest.mark.filterwarnings("ignore::DeprecationWarning")  # torch's own, on importing its compiler
@pytest.mark.parametrize("mode", ["plain", "seq", "states", "nobias"])
@pytest.mark.parametrize("how", ["run", "compile"])
def test_compiled_autograd(mode, how):
    """A backward captured as a graph, with the native node as a call of its own in it: run as it
    is, and traced and compiled further, where the node's backward goes through the op."""
    from torch._dynamo import compiled_autograd

    x, kw = _args(mode)
    dout = torch.randn_like(x).detach()
    dfinal = torch.randn(B, D, W - 1, device=DEV).to(x.dtype)
    want = _run(x, kw, dout, dfinal)
    captured, traced = [], []
    torch._dynamo.reset()  # (a backward captured before would be taken again)
    torch._C._dynamo.compiled_autograd.clear_cache()

    def note(gm, inputs):
        traced.extend(f"{n.target} {n.args}" for n in gm.graph.nodes)
        return make_boxed_func(gm.forward)

    def compiler(gm):
        captured.extend(str(n.target) for n in gm.graph.nodes)
        return gm if how == "run" else torch.compile(gm, backend=aot_autograd(fw_compiler=note))

    r = cc.causal_conv1d_fn(x, **kw)
    out, final = r if isinstance(r, tuple) else (r, None)
    ins = [t for t in (x, kw["weight"], kw["bias"], kw.get("initial_states")) if t is not None]
    outs, douts = ([out, final], [dout, dfinal]) if final is not None else ([out], [dout])
    with compiled_autograd._enable(compiler):
        torch.autograd.backward(outs, douts)
    got = [out, *([final] if final is not None else []), *(t.grad for t in ins)]
    assert any("Conv1dFn" in t for t in captured)
    assert how == "run" or any("_bwd_typed_inplace" in t for t in traced)
    for a, c in zip(got, want, strict=True):
        assert torch.equal(a.detach(), c.detach())
