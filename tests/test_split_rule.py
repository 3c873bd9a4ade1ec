"""Grad-hidden split counts of shapes outside the launch table (CPU, through
``orda_plan_info``): every split covers vocabulary rows, a split keeps at
least the rows the rule asks for, and the static entry still takes what at
most 16 splits would fit."""
from __future__ import annotations

import pytest

from orda_ce_kernel import _native

STATIC = 64 << 20


def _problem(dtype, N, H, V, chunk=0, splits=0):
    p = _native.Problem()
    p.abi_version = _native.ABI_VERSION
    p.mode, p.dtype, p.logits_dtype = 0, dtype, dtype
    p.n_rows, p.vocab, p.hidden, p.teacher_hidden = N, V, H, H
    p.ignore_index = -100
    f = _native.FLAG
    p.flags = (f["need_grad_student_hidden"] | f["need_grad_weight"] | f["grads_in_forward"] | f["compute_teacher_ce"]
               | f["compute_divergence"])
    p.temperature, p.student_ce_weight, p.teacher_ce_weight, p.kl_weight = 2.0, 1.0, 1.0, 1.0
    p.token_chunk, p.grad_hidden_splits = chunk, splits
    return p


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("N,H,V", [(1, 8, 5), (64, 64, 300), (256, 1024, 32000), (500, 520, 1023), (1999, 768, 50257),
                                   (512, 256, 4096), (4096, 4096, 100277), (8192, 64, 4096), (130, 2048, 152064)])
def test_splits_cover_the_vocabulary(dtype, N, H, V):
    info = _native.plan_info(_problem(dtype, N, H, V))
    sp = info["grad_hidden_splits"]
    assert 1 <= sp <= 64
    rows = -(-V // sp)
    assert sp == 1 or rows >= 192, (sp, rows)  # (K ranges are rounded up to 64 rows)


@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_static_entry_keeps_what_it_took(dtype):
    """Where the plan's own split count passes the static scratch, a call that
    fits with at most 16 splits is planned so."""
    seen = 0
    for N in (64, 128, 192, 256, 320, 384, 448, 512):
        for V in range(2000, 24000, 500):
            p = _problem(dtype, N, 1024, V)
            need = _native.forward_workspace_bytes(p)
            least = _native.forward_workspace_bytes(_problem(dtype, N, 1024, V, splits=8))
            if need > STATIC:
                assert _native.forward_workspace_bytes(_problem(dtype, N, 1024, V, splits=16)) > STATIC, (N, V)
            elif least > STATIC // 2:
                seen += 1
    assert seen > 0
