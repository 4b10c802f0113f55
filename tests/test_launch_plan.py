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
