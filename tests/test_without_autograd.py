"""Gradient recording off: the Functions see tensors that require no gradient
(a parameter inside ``Function.forward`` would still say so), and the caller's
own tensors are left as they are (CPU)."""
from __future__ import annotations

import pytest
import torch
import torch.autograd.forward_ad as fwd

from orda_ce_kernel.ops._engine import without_autograd


def test_tensors_are_detached_only_when_recording_is_off():
    w, x = torch.randn(4, 3, requires_grad=True), torch.randn(2, 3)
    assert without_autograd(w, x, None) == (w, x, None)
    with torch.no_grad():
        a, b, c = without_autograd(w, x, None)
    assert not a.requires_grad and not b.requires_grad and c is None
    assert a.data_ptr() == w.data_ptr() and a.shape == w.shape and w.requires_grad
    with torch.inference_mode():
        (d,) = without_autograd(w)
    assert not d.requires_grad and d.data_ptr() == w.data_ptr()


@pytest.mark.parametrize("requires_grad", [False, True])
def test_forward_mode_tangents_are_still_refused(requires_grad):
    """A Function without a jvp refuses dual tensors; so it does after this."""
    class Sum(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.sum()

        @staticmethod
        def backward(ctx, g):
            return g

    x = torch.randn(3, requires_grad=requires_grad)
    with fwd.dual_level(), torch.no_grad():
        (y,) = without_autograd(fwd.make_dual(x, torch.ones(3)))
        with pytest.raises(NotImplementedError):
            Sum.apply(y)
