"""Token counts off the kernels' quads, 256-token groups and 8-token padding,
and a short last token chunk, against the float64 oracle.  The workspace comes
from memory that holds NaN: padding columns of the chunk's logits are read by
the dlogits pass and must reach no gradient."""
from __future__ import annotations

import pytest
import torch

from tests.test_gpu_parity import _check, _close_grad, _grad_tol, _orda, _run

pytestmark = pytest.mark.gpu


def _poison(nbytes=96 << 20):
    """Free cached blocks full of NaN for the call's allocations to reuse."""
    for size in (nbytes, nbytes // 4, nbytes // 16, 1 << 20, 1 << 18):
        torch.full((size // 4,), float("nan"), device="cuda")
    torch.cuda.synchronize()


# one and two tokens, a partial quad, 256 + 1 .. + 3, one past the padding of
# 8; chunk 32 requests give chunks of 64 or 128 tokens, the last of 1 to 63
@pytest.mark.parametrize("N,chunk", [(1, None), (6, None), (255, None), (259, None), (513, None), (129, 32), (131, 32),
                                     (161, 32), (190, 32)])
@pytest.mark.parametrize("mode,dtype,V,div,T", [
    ("tied", torch.bfloat16, 1003, "forward_kl", 2.0), ("tied", torch.float32, 1000, "reverse_kl", 1.0),
    ("separate", torch.float16, 1030, "jsd", 2.0), ("separate", torch.float32, 517, "jsd", 2.0),
    ("precomputed_logits", torch.bfloat16, 1032, "forward_kl", 1.0),
    ("precomputed_logits", torch.bfloat16, 1032, "jsd", 2.0),
    ("precomputed_logits", torch.bfloat16, 1001, "hellinger", 1.0),
    ("precomputed_hidden", torch.bfloat16, 1027, "forward_kl", 4.0)])
def test_ragged_token_chunks(mode, dtype, V, div, T, N, chunk):
    o = _orda()
    _poison()
    print(f"[ragged] {mode} {dtype} N={N} V={V} chunk={chunk} {div}", flush=True)
    out, ref, hs, W, teacher = _run(
        mode, dtype, N=N, H=136, V=V, Ht=None if mode == "tied" else 72, seed=N + V, T=T, div=div,
        w_t=0.5 if mode == "separate" else None, ignore_frac=0.1 if N > 8 else 0.0, w_std=0.1,
        config=o.KernelConfig(chunk_size=chunk) if chunk else None)
    _check(out, ref, hs, W, dtype)
    if mode == "separate":
        for got, name in ((teacher.hidden, "grad_teacher_hidden"), (teacher.weight, "grad_teacher_weight")):
            _close_grad(got.grad, ref[name], name, _grad_tol(dtype))
