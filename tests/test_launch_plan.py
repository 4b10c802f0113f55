"""What the library launches, on the CPU: a spy takes the place of the HIP
runtime's launch call (``_launch_spy.py``), so the kernel of a call and the
memory that it is given can be checked without a GPU."""

from __future__ import annotations

import shutil

import pytest

import _launch_spy

pytestmark = pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc not installed")


def test_partial_sums_fit_into_the_workspace(tmp_path):
    """The records that a backward writes, and that its reduction reads, lie inside the
    workspace that cc1d_bwd_workspace_floats asks for: every length over several segments
    (both sides of each change in the vectors per lane), rows aligned, alike off the
    vector grid, unlike each other, channel-last with any channel count, and strided; under
    and over the 2048 rows at which the planner changes."""
    code = r"""
import random
rng = random.Random(0)
lengths = list(range(1, 5200)) + [rng.randint(5200, 20000) for _ in range(300)]
worst, kinds, bad = 0.0, {}, []
for dtype, es in ((1, 2), (2, 4)):
    places = {
        "tight": dict(),
        "alike, off the vector grid": dict(offsets=(es, es, es)),
        "unlike": dict(offsets=(0, es, 0)),
        "rows of a longer tensor": dict(pads=(3, 0, 0)),
        "channel-last": dict(layout="last"),
        "channel-last, odd rows": dict(layout="last", dim_pad=1),
        "strided": dict(layout="strided"),
    }
    for place, kw in places.items():
        for B, D in ((1, 63), (2, 1024)):
            if "last" in place or place == "strided":
                some = lengths[::17]
            else:
                some = lengths
            for L in some:
                for W in ((4,) if L % 7 else (2, 4, 5, 9)):
                    p = bwd_params(B, D, L, W, dtype, **kw)
                    need = lib.cc1d_bwd_workspace_floats(ctypes.byref(p))
                    status = bwd_typed(p)
                    if status != 0 or len(launches) != 2:
                        bad.append([place, dtype, B, D, L, W, "status", status])
                        continue
                    wrote, read = floats_touched()
                    k = launches[0][0]
                    kinds[k] = kinds.get(k, 0) + 1
                    if wrote > need or read > wrote:
                        bad.append([place, dtype, B, D, L, W, wrote, read, need])
                    if L % 64 == 0 and bwd_typed(p, need - 1) != 8:  # CC1D_ERR_WORKSPACE
                        bad.append([place, dtype, B, D, L, W, "a float less was taken"])
# the static scratch: at most its size, or refused
scratch = []
for D in (1000, 1049):  # 2 records of 5 floats a row: 2,000,000 and 2,098,000
    p = bwd_params(200, D, 3071, 4, 1)
    status = bwd_typed(p, 0, noalloc=True)
    scratch.append([status, floats_touched()[0] if status == 0 else 0])
result = {"kinds": kinds, "bad": bad[:40], "n_bad": len(bad), "scratch": scratch}
"""
    got = _launch_spy.run(code, tmp_path)
    assert set(got["kinds"]) == {"bwd_rows_vec", "bwd_rows_short", "bwd_clw", "bwd_generic"}, got["kinds"]
    assert got["n_bad"] == 0, got["bad"]
    assert got["scratch"] == [[0, 2_000_000], [9, 0]]  # CC1D_ERR_SCRATCH_LIMIT past 2,097,152


def test_an_empty_pool_takes_a_kernel_that_reads_no_row(tmp_path):
    """With no row in the pool every index is padding; update_dir, update_lin and update_step
    read row 0 in a padding entry's place, so such calls go to the generic kernel."""
    code = r"""
result = []
for dtype in (0, 1, 2):
    for W, S, state in ((4, 3, "line"), (4, 4, "line"), (9, 8, "line"), (4, 3, "step"), (9, 8, "step"), (4, 6, "step")):
        result.append([update(3, 64, W, dtype, S=S, state=state, rows=r, indices=True) for r in (5, 0)])
"""
    got = _launch_spy.run(code, tmp_path)
    assert {a for a, _ in got} == {"update_dir", "update_lin", "update_step"}
    assert {b for _, b in got} == {"update_generic"}


def test_channel_last_rows_of_whole_dwords_keep_their_own_kernel(tmp_path):
    """An even number of 16-bit channels on the dword grid takes the form of bwd_clw without the
    odd count's addresses (its last template argument), anything else the one with them."""
    code = r"""
result = []
for dtype, D, kw in ((1, 768, {}), (0, 4096, {}), (1, 769, {}), (1, 768, dict(dim_pad=1)), (0, 768, dict(offsets=(0, 2, 0))),
                     (2, 769, {})):
    for seq in (None, 1):
        p = bwd_params(2, D, 512, 4, dtype, layout="last", seq_stride=seq, **kw)
        assert bwd_typed(p) == 0
        result.append([launches[0][0], template_values(launches[0][5])[-1]])
"""
    got = _launch_spy.run(code, tmp_path)
    assert {k for k, _ in got} == {"bwd_clw"}
    assert [odd for _, odd in got] == [0, 0, 0, 0, 1, 1, 1, 1, 1, 1, 0, 0]


def test_kernel_of_each_layout(tmp_path):
    """Which kernel a call takes, forward and backward, by length, type and layout (RowsMode 0:
    aligned, 1: alike, 2: any), and a decode update by its state."""
    code = r"""
bf16, fp32 = 1, 2

def both(L, dtype=bf16, B=4, D=512, W=4, seq=False, **kw):
    fkw = {k: v[:2] if k in ("offsets", "pads") else v for k, v in kw.items()}
    p = bwd_params(B, D, L, W, dtype, seq_stride=1 if seq else None, **kw)
    assert bwd_typed(p) == 0
    b = route(launches[0])
    return [fwd(B, D, L, W, dtype, seq=seq, **fkw), b]

result = {
    "aligned": both(2048), "aligned with ids": both(2048, seq=True), "aligned fp32": both(2048, fp32),
    "odd length": both(2041), "odd length, a vector more": both(1023), "odd length fp32": both(1023, fp32),
    "no more segments than the aligned form": [both(L, D=48, B=2)[1] for L in (3071, 5119)],
    "unlike": both(2048, offsets=(2, 4, 6)), "unlike rows": both(2041, pads=(1, 2, 3)),
    "unlike fp32": both(2048, fp32, offsets=(4, 8, 12)),
    "32 vectors": both(256), "33 vectors": both(264), "short, unlike": both(100, pads=(1, 2, 3)),
    "channel-last": both(2048, layout="last"), "channel-last, odd": both(2048, D=513, layout="last"),
    "one channel": both(2048, D=1, layout="last", dim_pad=7, dtype=bf16),
    "strided": both(2048, layout="strided"), "fp32 width 9": both(2048, fp32, W=9),
    "update": [update(8, 512, 4, bf16, S=3), update(8, 512, 4, bf16, S=4), update(8, 512, 9, bf16, S=8),
               update(8, 512, 4, bf16, S=3, state="step"), update(8, 512, 4, bf16, S=6),
               update(8, 512, 4, bf16, S=64, ring=True), update(256, 5120, 4, bf16, S=64, ring=True),
               update(8, 512, 4, bf16, S=64, ring=True, tokens=8), update(8, 512, 4, bf16, S=63, ring=True)],
}
"""
    got = _launch_spy.run(code, tmp_path)

    def rows(f, b):
        return [["fwd_rows_vec", f], ["bwd_rows_vec", b]]

    short = [["fwd_rows_short", None], ["bwd_rows_short", None]]
    last = [["fwd_cl", None], ["bwd_clw", None]]
    generic = [["fwd_generic", None], ["bwd_generic", None]]
    assert got == {
        "aligned": rows(0, 0), "aligned with ids": rows(0, 0), "aligned fp32": rows(0, 0),
        "odd length": rows(1, 1), "odd length, a vector more": rows(2, 2), "odd length fp32": rows(1, 1),
        "no more segments than the aligned form": [["bwd_rows_vec", 1]] * 2,
        "unlike": rows(2, 2), "unlike rows": rows(2, 2), "unlike fp32": rows(2, 2),
        "32 vectors": short, "33 vectors": rows(0, 0), "short, unlike": short,
        "channel-last": last, "channel-last, odd": last, "one channel": generic,
        "strided": generic, "fp32 width 9": generic,
        "update": ["update_dir", "update_dir", "update_lin", "update_step", "update_generic", "update_circ_vec",
                   "update_ring", "update_ring", "update_circ"],
    }
