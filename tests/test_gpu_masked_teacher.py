"""Cached 16-bit teacher logits that are -inf (or the type's lowest value) over
a stretch of the vocabulary: no probability there, and the losses and gradients
of the rest as the float64 oracle has them.

The stretches cover the first tile of a vocabulary range whose later tiles are
finite (600 tokens x 32000: two 256-row tiles to a range in the losses-only
scan; 2100 x 20000: three), all of a lane's rows within it (116 rows), and ends
of the vocabulary; vocabulary 32003 takes the two-stage engine.  Losses come
from fp32 accumulators of 16-bit operands (1e-5), gradients are rounded to 16
bits and their operands too: 2^-8 (bf16) / 2^-11 (fp16) of their norm each,
2e-2 / 5e-3 with the tails."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.orda_oracle import distillation_loss_oracle
from tests.test_gpu_parity import _make, _np, _orda

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("value", ["inf", "lowest"])
@pytest.mark.parametrize("dtype,div", [(torch.bfloat16, "hellinger"), (torch.float16, "tvd"), (torch.float16, "hellinger")])
@pytest.mark.parametrize("N,V,stretches", [(600, 32000, [(0, 256), (2048, 140)]), (2100, 20000, [(0, 700), (15360, 256)]),
                                           (600, 32003, [(0, 512), (31000, 1003)]), (130, 4096, [(0, 300)])])
def test_masked_stretch_of_cached_logits(N, V, stretches, dtype, div, value, train):
    o = _orda()
    H = 128
    hs, ht, W, Wt, y = _make(N, N, H, V, dtype, w_std=1.5 / H ** 0.5, ignore_frac=0.1)
    lt = (ht.float() @ Wt.float().t()).to(dtype)
    low = -torch.inf if value == "inf" else torch.finfo(dtype).min
    masked = torch.zeros(V, dtype=torch.bool)
    for start, length in stretches:
        masked[start:start + length] = True
    lt[:, masked] = low
    hs_d, W_d = hs.cuda().requires_grad_(train), W.cuda().requires_grad_(True)
    print(f"[masked] N={N} V={V} {div} {value} train={train}", flush=True)
    with torch.set_grad_enabled(train):
        out = o.distillation_loss(hs_d, W_d, y.cuda(), o.PrecomputedTeacher(logits=lt.cuda()), student_ce_weight=0.5,
                                  kl_weight=0.5, divergence=div, backend="hip")
    far = _np(lt)
    far[:, masked.numpy()] = -1e4  # probability 0 in float64 too
    ref = distillation_loss_oracle("precomputed", _np(hs), _np(W), y.numpy(), teacher_logits=far, student_ce_weight=0.5,
                                   kl_weight=0.5, divergence=div)
    for name in ("loss", "student_ce", "kl"):
        got = float(getattr(out, name))
        tol = 2e-5 if not train else 1e-4  # (training stores the student's logits in 16 bits for a two-pass divergence)
        assert np.isfinite(got) and abs(got - ref[name]) <= tol + tol * abs(ref[name]), f"{name}: {got} against {ref[name]}"
    if not train:
        return
    out.loss.backward()
    tol = 2e-2 if dtype == torch.bfloat16 else 5e-3
    if div == "tvd":  # its gradient jumps where p_s = p_t, which a rounded logit can cross
        tol *= 2
    for got, want in ((hs_d.grad, ref["grad_student_hidden"]), (W_d.grad, ref["grad_weight"])):
        got = _np(got)
        assert np.all(np.isfinite(got))
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
