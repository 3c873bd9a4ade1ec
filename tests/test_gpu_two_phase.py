"""The two-phase backward (fp32-accumulated weight gradients): vocabulary
chunks, a ragged last chunk with fewer splits, token counts off the padding,
every teacher mode and gradient, against the float64 oracle and (16-bit)
against the error of one rounding: each gradient is one fp32 sum rounded once,
its operands the dlogits rounded to 16 bits, so it is off by at most 2^-8
(bf16) or 2^-11 (fp16) of its norm from the rounding of the operands and
again from its own: 2e-2 and 5e-3 leave room for the tails."""
from __future__ import annotations

import pytest
import torch

from tests.test_gpu_parity import _check, _close_grad, _grad_tol, _orda, _run
from tests.test_gpu_ragged_chunks import _poison

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,V,chunks", [(1, 8, 5, 1), (7, 72, 300, 2), (65, 136, 515, 2), (130, 264, 1030, 3),
                                          (257, 64, 4099, 8), (600, 520, 2050, 4)])
@pytest.mark.parametrize("mode,dtype,div,T,w_t", [
    ("tied", torch.bfloat16, "forward_kl", 2.0, 0.6), ("tied", torch.float16, "jsd", 1.0, 0.6),
    ("tied", torch.bfloat16, "reverse_kl", 1.0, 0.0), ("tied", torch.float32, "forward_kl", 1.0, 0.6),
    ("separate", torch.bfloat16, "forward_kl", 2.0, None), ("separate", torch.float16, "hellinger", 2.0, 0.5),
    ("separate", torch.float32, "jsd", 2.0, 0.5), ("precomputed_logits", torch.bfloat16, "skew_reverse_kl", 1.0, None),
    ("precomputed_hidden", torch.bfloat16, "reverse_kl", 4.0, None)])
def test_two_phase_matches_oracle(mode, dtype, div, T, w_t, N, H, V, chunks):
    o = _orda()
    _poison()
    print(f"[two-phase] {mode} {dtype} {div} N={N} H={H} V={V} chunks={chunks}", flush=True)
    cfg = o.KernelConfig(fp32_grad_weight_accumulation=True, num_chunks=min(chunks, N))
    out, ref, hs, W, teacher = _run(mode, dtype, N=N, H=H, V=V, Ht=None if mode == "tied" else H + 8, seed=N, T=T,
                                    div=div, w_t=w_t, config=cfg, w_std=1.5 / H ** 0.5, grad_output=1.5,
                                    ignore_frac=0.1 if N > 8 else 0.0, grad_teacher=bool(w_t) or mode != "separate")
    _check(out, ref, hs, W, dtype)
    if mode in ("tied", "separate") and w_t:
        _close_grad(teacher.hidden.grad, ref["grad_teacher_hidden"], "grad_teacher_hidden", _grad_tol(dtype))
    if mode == "separate" and w_t:
        _close_grad(teacher.weight.grad, ref["grad_teacher_weight"], "grad_teacher_weight", _grad_tol(dtype))
