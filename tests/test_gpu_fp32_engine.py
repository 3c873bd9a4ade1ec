"""The fp32 kernels (three-way bf16 split on the matrix cores) at the edges of
their tiles, against the float64 oracle.

Bound: an fp32 value is the sum of its three parts and the dropped products are
below 2^-24 |a b|, so a dot product of K terms is off by at most (6 K / 32 + 1)
2^-24 sum |a b| (one rounding per 32-term MFMA and product; far less where the
roundings' signs mix).  With
K <= 600, logits of spread 1.5 and the softmax's exp on 2^-23 accurate
hardware, losses and gradients agree to 1e-5 of their norm (1e-6 seen)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.test_gpu_parity import _make, _np, _orda, _run
from oracle.orda_oracle import distillation_loss_oracle

pytestmark = pytest.mark.gpu


def _close(got, want, name, tol=1e-5):
    got = np.asarray(got.detach().double().cpu())
    assert np.all(np.isfinite(got)), name
    err = np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30)
    assert err <= tol, f"{name}: {err:.2e}"


# 64- and 128-token scan tiles, 256-row vocabulary tiles, 64- and 128-wide GEMM
# tiles and 32-wide K steps, each one short of, at and past its edge; the last
# shapes fill the large tiles (256 x 128, a workgroup per CU)
SHAPES = [(1, 4, 255), (63, 36, 257), (65, 128, 300), (129, 132, 513), (200, 260, 1000), (127, 31 * 4, 4097),
          (520, 600, 12000)]


@pytest.mark.parametrize("N,H,V", SHAPES)
@pytest.mark.parametrize("mode,div,T,w_t", [("tied", "forward_kl", 2.0, 0.7), ("tied", "jsd", 1.0, 0.0),
                                            ("separate", "reverse_kl", 1.0, 0.5),
                                            ("precomputed_logits", "hellinger", 2.0, None),
                                            ("precomputed_hidden", "squared_l2", 1.0, None)])
def test_fp32_tile_edges(mode, div, T, w_t, N, H, V):
    print(f"[fp32] {mode} {div} N={N} H={H} V={V}", flush=True)
    out, ref, hs, W, teacher = _run(mode, torch.float32, N=N, H=H, V=V, Ht=H if mode == "tied" else H + 40, seed=N,
                                    T=T, div=div, w_t=w_t, w_std=1.5 / H ** 0.5, ignore_frac=0.1 if N > 8 else 0.0)
    for name in ("loss", "student_ce", "kl"):
        assert abs(float(getattr(out, name)) - ref[name]) <= 1e-6 + 1e-5 * abs(ref[name]), name
    _close(hs.grad, ref["grad_student_hidden"], "grad_student_hidden")
    _close(W.grad, ref["grad_weight"], "grad_weight")
    if mode == "separate":
        _close(teacher.hidden.grad, ref["grad_teacher_hidden"], "grad_teacher_hidden")
        _close(teacher.weight.grad, ref["grad_teacher_weight"], "grad_teacher_weight")


@pytest.mark.parametrize("mode", ["tied", "separate"])
def test_fp32_operands_of_unequal_scale(mode):
    """Columns of the hidden states scaled by 2^12 and of the weight by 2^-12
    (and the reverse): the products cancel the scales, each operand's parts
    span 24 bits more."""
    o = _orda()
    N, H, V = 150, 96, 700
    hs, ht, W, Wt, y = _make(5, N, H, V, torch.float32, w_std=1.5 / H ** 0.5)
    s = torch.tensor([2.0 ** 12, 2.0 ** -12]).repeat(H // 2)
    hs, ht, W, Wt = hs * s, ht * s, W / s, Wt / s
    hs_d, W_d = hs.cuda().requires_grad_(True), W.cuda().requires_grad_(True)
    teacher = o.TiedTeacher(ht.cuda()) if mode == "tied" else o.SeparateTeacher(ht.cuda(), Wt.cuda())
    out = o.distillation_loss(hs_d, W_d, y.cuda(), teacher, teacher_ce_weight=0.0, kl_weight=0.5, backend="hip")
    out.loss.backward()
    ref = distillation_loss_oracle(mode, _np(hs), _np(W), y.numpy(), teacher_hidden=_np(ht), teacher_ce_weight=0.0,
                                   teacher_weight=None if mode == "tied" else _np(Wt), kl_weight=0.5)
    assert abs(float(out.loss) - ref["loss"]) <= 1e-5 * abs(ref["loss"])
    _close(hs_d.grad, ref["grad_student_hidden"], "grad_student_hidden")
    _close(W_d.grad, ref["grad_weight"], "grad_weight")


@pytest.mark.parametrize("div", ["hellinger", "tvd"])
@pytest.mark.parametrize("start,length", [(0, 64), (37, 130), (600, 400)])
def test_fp32_masked_stretch_of_teacher_logits(div, start, length):
    """Teacher logits that are -inf over a stretch of the vocabulary longer
    than a lane's rows of a tile carry no probability there."""
    o = _orda()
    N, H, V = 70, 32, 1000
    hs, ht, W, Wt, y = _make(9, N, H, V, torch.float32, w_std=0.3)
    lt = ht @ Wt.t()
    lt[:, start:start + length] = -torch.inf
    hs_d, W_d = hs.cuda().requires_grad_(True), W.cuda().requires_grad_(True)
    out = o.distillation_loss(hs_d, W_d, y.cuda(), o.PrecomputedTeacher(logits=lt.cuda()), kl_weight=0.5,
                              divergence=div, backend="hip")
    far = lt.double().masked_fill(torch.isinf(lt), -1e4).numpy()  # probability 0 in float64 too
    ref = distillation_loss_oracle("precomputed", _np(hs), _np(W), y.numpy(), teacher_logits=far, kl_weight=0.5,
                                   divergence=div)
    assert abs(float(out.kl) - ref["kl"]) <= 1e-6 + 1e-5 * abs(ref["kl"])
    out.loss.backward()
    _close(W_d.grad, ref["grad_weight"], "grad_weight", 1e-5 if div == "hellinger" else 1e-3)
