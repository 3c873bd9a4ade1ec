"""Evaluation passes (``torch.no_grad()`` with parameters that require a
gradient) against the float64 oracle.

The losses come from fp32 accumulators of 16-bit operands: products are exact
in fp32, so a logit of K terms is off by at most K 2^-24 sum|h w| (2e-5 here),
which the softmax averages: losses within 1e-5 relative, plus 2e-5 absolute
for values near zero.  Logits of a cached teacher are exact inputs."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.orda_oracle import distillation_loss_oracle
from tests.test_gpu_parity import _make, _np, _orda

pytestmark = pytest.mark.gpu


# 256-token and 128-token tiles, 256-row vocabulary tiles: one token, a ragged
# last tile, exact tiles; hidden sizes at the ring engine's limit (64 is the
# two-stage engine's); vocabularies off 4, off 8 and off 256
SHAPES = [(1, 72, 257), (129, 64, 1000), (255, 128, 1028), (512, 200, 2048), (300, 96, 1030), (257, 136, 4099)]


@pytest.mark.parametrize("N,H,V", SHAPES)
@pytest.mark.parametrize("div,T", [("forward_kl", 1.0), ("reverse_kl", 2.0), ("jsd", 2.0), ("hellinger", 1.0),
                                   ("squared_l2", 2.0)])
@pytest.mark.parametrize("mode", ["tied", "separate", "logits", "none"])
def test_no_grad_losses_match_the_oracle(mode, div, T, N, H, V):
    o = _orda()
    dtype = torch.bfloat16 if (N + V) % 2 else torch.float16
    hs, ht, W, Wt, y = _make(N + V, N, H, V, dtype, Ht=H if mode == "tied" else H + 8, ignore_frac=0.1,
                             w_std=1.5 / H ** 0.5)
    if N == 1:
        y[:] = 3
    w_kl, w_t = (0.0, 0.0) if mode == "none" else (0.8, 0.6 if mode in ("tied", "separate") else 0.0)
    if mode == "tied":
        teacher, kw = o.TiedTeacher(ht.cuda().requires_grad_(True)), dict(teacher_hidden=_np(ht))
    elif mode == "separate":
        teacher = o.SeparateTeacher(ht.cuda(), Wt.cuda().requires_grad_(True))
        kw = dict(teacher_hidden=_np(ht), teacher_weight=_np(Wt))
    else:
        lt = (ht.float() @ Wt.float().t()).to(dtype)
        teacher, kw = o.PrecomputedTeacher(logits=lt.cuda()), dict(teacher_logits=_np(lt))
    W_d = W.cuda().requires_grad_(True)
    print(f"[eval] {mode} {div} N={N} H={H} V={V}", flush=True)
    with torch.no_grad():
        out = o.distillation_loss(hs.cuda(), W_d, y.cuda(), teacher, student_ce_weight=0.7, teacher_ce_weight=w_t,
                                  kl_weight=w_kl, kl_temperature=T, divergence=div, backend="hip")
    assert not out.loss.requires_grad and W_d.grad is None
    ref = distillation_loss_oracle(
        "precomputed" if mode in ("logits", "none") else mode, _np(hs), _np(W), y.numpy(), student_ce_weight=0.7,
        teacher_ce_weight=w_t, kl_weight=w_kl, kl_temperature=T, divergence=div, **kw)
    for name in ("loss", "student_ce", "teacher_ce", "kl"):
        got = float(getattr(out, name))
        want = ref[name] if (name != "kl" or w_kl) else 0.0
        assert np.isfinite(got) and abs(got - want) <= 2e-5 + 1e-5 * abs(want), f"{name}: {got} against {want}"
