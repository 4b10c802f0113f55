"""The native host path without a GPU: it loads, and leaves every call that is not its own to the Python code."""

from __future__ import annotations

import pytest
import torch

from causal_conv1d_amd import _host


def test_cpu_tensors_and_odd_arguments_are_left_to_python():
    ext = _host.load()
    x, w = torch.randn(2, 4, 8), torch.randn(4, 4)
    for args in ((x, w, None, None, None, False, None, "silu"), (x, w, None, None, None, False, None, "relu"),
                 (None, w, None, None, None, False, None, None), ("x", 3, None, None, None, 1, None, None)):
        assert ext.fn(*args) is NotImplemented
    assert ext.update(x, torch.zeros(2, 4, 3), w, None, None, None, None) is NotImplemented
    assert ext.varlen_states(x[0], torch.tensor([0, 2], dtype=torch.int32), 3) is NotImplemented
    for f, n in ((ext.fn, 8), (ext.update, 7), (ext.varlen_states, 3), (ext.bind, 6)):
        with pytest.raises(RuntimeError, match=f"takes {n}"):
            f(x)
