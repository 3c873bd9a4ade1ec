"""Plans at the ends of the stated sizes (CPU, through the library's planning
entries): n_rows and vocab up to 2^30, hidden up to 2^22."""
from __future__ import annotations

import pytest

from orda_ce_kernel import _native

BF16, F16, F32 = 0, 1, 2


def _problem(mode="tied", dtype=BF16, N=512, H=256, V=4096, Ht=None, flags=(), logits_dtype=None, div=0):
    p = _native.Problem()
    p.abi_version = _native.ABI_VERSION
    p.mode, p.dtype, p.logits_dtype = _native.MODE[mode], dtype, dtype if logits_dtype is None else logits_dtype
    p.n_rows, p.vocab, p.hidden, p.teacher_hidden = N, V, H, H if Ht is None else Ht
    p.ignore_index = -100
    for name in flags:
        p.flags |= _native.FLAG[name]
    p.divergence = div
    p.temperature, p.student_ce_weight, p.teacher_ce_weight, p.kl_weight = 2.0, 1.0, 1.0, 1.0
    return p


GRADS = ("need_grad_student_hidden", "need_grad_weight", "compute_teacher_ce", "compute_divergence")


@pytest.mark.parametrize("dtype,N,H,V,flags", [
    (BF16, 1 << 23, 64, 4096, GRADS + ("grads_in_forward",)), (F32, 1 << 22, 64, 4096, GRADS + ("grads_in_forward",)),
    (BF16, (1 << 24) + 64, 64, 4096, ("compute_divergence",)), (F32, (1 << 23) + 64, 64, 4096, ("compute_divergence",)),
    (BF16, 1 << 30, 64, 4096, ()), (BF16, 64, 131072, 600000, ("compute_divergence",)),
    (BF16, 64, 131072, 600000, GRADS), (F32, 64, 131072, 600000, GRADS),
    (F16, (1 << 24) + 64, 64, 4096, ("need_grad_student_hidden",)),
    (BF16, 64, 131072, 600000, ("need_grad_weight",))])
def test_large_calls_are_planned(dtype, N, H, V, flags):
    """A limit of the grad-hidden GEMM's split ranges does not refuse calls that
    run without that GEMM, nor two-phase ones, whose general kernel has none."""
    p = _problem(dtype=dtype, N=N, H=H, V=V, flags=flags)
    assert _native.forward_workspace_bytes(p) > 0
    assert _native.saved_bytes(p) > 0
    assert "grads_in_forward" in flags or _native.backward_workspace_bytes(p) > 0


@pytest.mark.parametrize("dtype", [BF16, F32])
def test_cached_logits_need_no_teacher_hidden_size(dtype):
    """Teacher logits come without a hidden size; also a plan past the static
    scratch, which is planned again with fewer splits, divides by none."""
    p = _problem("precomputed_logits", dtype, N=1024, H=512, V=60000, Ht=0,
                 flags=("need_grad_student_hidden", "need_grad_weight", "compute_divergence", "grads_in_forward"))
    assert _native.forward_workspace_bytes(p) > 64 << 20
    assert _native.plan_info(p)["grad_hidden_splits"] >= 1


@pytest.mark.parametrize("N,H,V", [(32768, 5120, 152064), (8192, 4096, 128256)])
def test_two_phase_workspace_holds_one_fp32_sum(N, H, V):
    """A grad-hidden GEMM of one split needs one fp32 [N x H] sum over the
    vocabulary chunks beside the transposed rows and 512 MiB of dlogits."""
    p = _problem(N=N, H=H, V=V, flags=GRADS)
    got = _native.backward_workspace_bytes(p)
    assert got <= 4 * N * H + 2 * 2 * N * H + (512 << 20) + (1 << 20), got / 2 ** 20


def test_fp32_hidden_sizes_past_a_resource():
    """2^22 for the split-operand engine (256 rows in a resource of 4 GiB); the
    two-phase backward's two-stage kernel has 2 GiB, so half of that."""
    wide = dict(dtype=F32, N=64, H=1 << 22, V=1024)
    assert _native.forward_workspace_bytes(_problem(flags=("compute_divergence",), **wide)) > 0
    assert _native.forward_workspace_bytes(_problem(flags=GRADS + ("grads_in_forward",), **wide)) > 0
    with pytest.raises(ValueError, match="two-phase"):
        _native.forward_workspace_bytes(_problem(flags=GRADS, **wide))
    wide["H"] = 1 << 21
    assert _native.backward_workspace_bytes(_problem(flags=GRADS, **wide)) > 0


@pytest.mark.parametrize("dtype,most", [(BF16, 8388600), (F16, 8388600), (F32, 4194296)])
def test_two_phase_weight_gradient_of_too_many_tokens_is_refused(dtype, most):
    """Its K-major rows of tokens stay inside a buffer resource; past it they
    would wrap around."""
    flags = ("need_grad_weight", "compute_divergence")
    assert _native.backward_workspace_bytes(_problem(dtype=dtype, N=most, H=64, V=512, flags=flags)) > 0
    with pytest.raises(ValueError, match="tokens"):
        _native.forward_workspace_bytes(_problem(dtype=dtype, N=most + 1, H=64, V=512, flags=flags))
    with pytest.raises(ValueError, match="tokens"):
        _native.forward_workspace_bytes(_problem(dtype=dtype, N=most // 2 + 8, H=64, V=512,
                                                 flags=flags + ("compute_teacher_ce",)))


TIED = ("compute_teacher_ce", "compute_divergence")
STUDENT_GRADS = ("need_grad_student_hidden", "need_grad_weight", "grads_in_forward")


# (workgroups: token tiles times vocabulary ranges of whole 256-row tiles, as
# many ranges as keep them within 256 -- 2048 for the two-stage forward)
@pytest.mark.parametrize("mode,dtype,N,H,V,flags,engine,tokens,groups", [
    ("tied", F32, 512, 256, 4096, TIED + STUDENT_GRADS, 2, 64, 8 * 16),
    ("tied", F32, 512, 256, 4096, TIED, 2, 64, 8 * 16), ("separate", F32, 512, 256, 4096, TIED, 2, 64, 8 * 16),
    ("separate", F32, 512, 256, 4096, ("compute_divergence",) + STUDENT_GRADS, 2, 128, 4 * 16),
    ("precomputed_logits", F32, 512, 256, 4096, ("compute_divergence",), 2, 128, 4 * 16),
    ("tied", BF16, 4096, 4096, 128256, (), 1, 256, 16 * 16), ("tied", BF16, 4096, 64, 4096, (), 0, 128, 32 * 16),
    ("tied", BF16, 512, 4096, 4096, TIED, 1, 128, 4 * 16), ("separate", F16, 512, 256, 4096, TIED, 0, 128, 4 * 16),
    ("precomputed_logits", F16, 512, 256, 4096, ("compute_divergence",), 1, 256, 2 * 16),
    ("precomputed_logits", F16, 512, 256, 4098, ("compute_divergence",), 0, 128, 4 * 17)])
def test_plan_info_names_the_scan_that_runs(mode, dtype, N, H, V, flags, engine, tokens, groups):
    info = _native.plan_info(_problem(mode, dtype, N, H, V, flags=flags))
    assert (info["scan_engine"], info["scan_tokens_per_tile"], info["scan_workgroups"]) == (engine, tokens, groups)
