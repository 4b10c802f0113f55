"""Records the launches of libcc1d_amd.so without a GPU: which kernel a call
takes, with what grid and arguments. ``run`` executes a test's code in a fresh
process that loads ``launch_spy.c`` ahead of the HIP runtime (no torch there: it
brings the runtime with it); the code uses what this module defines."""

from __future__ import annotations

import ctypes
import importlib.util
import json
import re
import subprocess
import sys
from pathlib import Path

TESTS = Path(__file__).resolve().parent
_LIB_PY = TESTS.parent / "causal-conv1d-mojo_amd" / "causal_conv1d_amd" / "_lib.py"
FAKE = 1 << 24  # a 16-byte aligned address that nobody reads


def run(code: str, tmp_path):
    """What ``code`` leaves in ``result`` (plain values), executed with this module's names."""
    spy = tmp_path / "launch_spy.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(TESTS / "launch_spy.c"), "-o", str(spy)], check=True)
    prog = (f"import json, sys\nsys.path.insert(0, {str(TESTS)!r})\nimport _launch_spy\n_launch_spy.setup({str(spy)!r})\n"
            f"from _launch_spy import *\n{code}\nprint('RESULT ' + json.dumps(result))\n")
    res = subprocess.run([sys.executable, "-c", prog], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stderr
    return json.loads(res.stdout.rsplit("RESULT ", 1)[1])


# ---- in the fresh process ----

_spec = importlib.util.spec_from_file_location("_lib", _LIB_PY)
_lib = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(_lib)

_i64, _i32, _u32, _vp = ctypes.c_int64, ctypes.c_int32, ctypes.c_uint32, ctypes.c_void_p


class BwdArgs(ctypes.Structure):  # csrc/cc1d_bwd_kernels.hpp
    _fields_ = [("p", _lib.BwdParams), ("nseg_div", _u32 * 3), ("dim_div", _u32 * 3), ("part", _vp), ("nseg", _i64),
                ("n_items", _i64), ("chunk", _i64), ("groups", _i64), ("nvec", _i32)]


class RedArgs(ctypes.Structure):
    _fields_ = [("part", _vp), ("dweight", _vp), ("dbias", _vp), ("dweight_stride", _i64 * 2), ("dbias_stride", _i64),
                ("batch", _i64), ("dim", _i64), ("nseg", _i64), ("groups", _i64), ("nc", _i32), ("nout", _i64)]


lib = None
launches: list = []  # (kernel, grid x, grid y, block x, struct of its argument or None, mangled name)
_keep: list = []


def _name(mangled: str) -> str:
    """The kernel's plain name: the identifier in namespace cc1d."""
    m = re.match(r"_ZN4cc1d(?:12_GLOBAL__N_1)?(\d+)", mangled)
    return mangled[m.end():m.end() + int(m.group(1))]


def template_values(mangled: str) -> list[int]:
    """The integer and boolean template arguments, in order."""
    return [int(v) for v in re.findall(r"L[ib](\d+)E", mangled)]


def setup(spy_path: str) -> None:
    global lib
    spy = ctypes.CDLL(spy_path, mode=ctypes.RTLD_GLOBAL)
    cb_type = ctypes.CFUNCTYPE(None, ctypes.c_char_p, _u32, _u32, _u32, ctypes.POINTER(_vp))

    def on_launch(name, gx, gy, bx, args):
        mangled = name.decode()
        kernel = _name(mangled)
        arg = None
        if kernel.startswith("bwd_reduce"):
            arg = RedArgs.from_buffer_copy(ctypes.string_at(args[0], ctypes.sizeof(RedArgs)))
        elif kernel.startswith("bwd_"):
            arg = BwdArgs.from_buffer_copy(ctypes.string_at(args[0], ctypes.sizeof(BwdArgs)))
        launches.append((kernel, gx, gy, bx, arg, mangled))

    _keep.extend((spy, cb_type(on_launch)))
    spy.spy_callback(_keep[-1])
    lib = _lib.load()


def _strides(layout, D, L, pad, dim_pad):
    if layout == "rows":
        return D * (L + pad), L + pad, 1
    if layout == "last":
        return L * (D + dim_pad), 1, D + dim_pad
    return 2 * D * L, 2 * L, 2  # no unit stride


def bwd_params(B, D, L, W, dtype, *, layout="rows", offsets=(0, 0, 0), pads=(0, 0, 0), seq_stride=None, dim_pad=0):
    """cc1d_bwd_params of tensors that lie as said: byte offsets and row pads (elements) of x, dout and dx."""
    p = _lib.BwdParams()
    p.x, p.dout, p.dx = (FAKE + o for o in offsets)
    p.weight, p.bias = FAKE, FAKE
    p.batch, p.dim, p.seqlen, p.width, p.dtype, p.apply_silu = B, D, L, W, dtype, 1
    for stride, pad in zip((p.x_stride, p.dout_stride, p.dx_stride), pads):
        stride[:] = _strides(layout, D, L, pad, dim_pad)
    p.weight_stride[:] = (W, 1)
    p.bias_stride = 1
    if seq_stride is not None:
        p.seq_idx = FAKE
        p.seq_idx_stride[:] = (L * seq_stride, seq_stride)
    return p


def bwd_typed(p, floats=None, noalloc=False):
    """Status of the typed backward with a workspace of ``floats`` (default: what the library asks for)."""
    launches.clear()
    g = _lib.BwdGrads()
    g.dweight, g.dbias, g.workspace = FAKE, FAKE, FAKE
    g.dweight_stride[:] = (p.width, 1)
    g.dbias_stride = 1
    g.workspace_floats = lib.cc1d_bwd_workspace_floats(ctypes.byref(p)) if floats is None else floats
    f = lib.cc1d_bwd_typed_noalloc if noalloc else lib.cc1d_bwd_typed
    return f(ctypes.byref(p), ctypes.byref(g), None)


def floats_touched():
    """Floats of the workspace that the two launches of the last typed backward write and read."""
    (kernel, gx, _, _, a, _), (red, _, _, _, r, _) = launches
    assert red.startswith("bwd_reduce"), red
    W = a.p.width
    if kernel == "bwd_clw":
        channels = 64 * (1 if a.p.dtype == 2 else 2)
        wrote = gx * channels * (W + 1)
        read = r.batch * r.nseg * r.groups * r.nc * (W + 1)
    else:
        wrote = a.n_items * (W + 1)
        read = r.batch * r.nseg * r.dim * (W + 1)
    return wrote, read


def fwd(B, D, L, W, dtype, *, layout="rows", offsets=(0, 0), pads=(0, 0), seq=False, dim_pad=0):
    """Kernel of a forward, and its RowsMode (None unless fwd_rows_vec)."""
    launches.clear()
    p = _lib.FwdParams()
    p.x, p.out = (FAKE + o for o in offsets)
    p.weight, p.bias = FAKE, FAKE
    p.batch, p.dim, p.seqlen, p.width, p.dtype, p.apply_silu = B, D, L, W, dtype, 1
    for stride, pad in zip((p.x_stride, p.out_stride), pads):
        stride[:] = _strides(layout, D, L, pad, dim_pad)
    p.weight_stride[:] = (W, 1)
    p.bias_stride = 1
    if seq:
        p.seq_idx = FAKE
        p.seq_idx_stride[:] = (L, 1)
    status = lib.cc1d_fwd(ctypes.byref(p), None)
    assert status == 0 and len(launches) == 1, status
    return route(launches[0])


def route(launch):
    """[kernel, RowsMode of a *_rows_vec kernel or None]"""
    return [launch[0], template_values(launch[5])[-1] if launch[0].endswith("rows_vec") else None]


def update(B, D, W, dtype, *, S, state="line", rows=None, tokens=1, ring=False, indices=False):
    """Kernel of a decode update: state rows of lines (a channel's S values together) or steps."""
    launches.clear()
    p = _lib.UpdateParams()
    p.x, p.weight, p.bias, p.conv_state, p.out = (FAKE,) * 5
    p.conv_state_indices = FAKE if indices else None
    p.cache_seqlens = FAKE if ring else None
    p.batch, p.dim, p.seqlen, p.width, p.state_len = B, D, tokens, W, S
    p.state_rows = B if rows is None else rows
    p.x_stride[:] = p.out_stride[:] = (D * tokens, tokens, 1)
    p.weight_stride[:] = (W, 1)
    p.bias_stride = 1
    p.conv_state_stride[:] = (D * S, S, 1) if state == "line" else (D * S, 1, D)
    p.dtype, p.apply_silu = dtype, 1
    status = lib.cc1d_update(ctypes.byref(p), None)
    assert status == 0 and len(launches) == 1, status
    return launches[0][0]


__all__ = ["lib", "launches", "bwd_params", "bwd_typed", "floats_touched", "template_values", "route", "fwd", "update",
           "ctypes", "_lib", "FAKE"]
