"""fp32 operands without a three-way bf16 split (infinities, magnitudes that
round past the bf16 range) and short sums, where the split-operand engine takes
the native fp32 MFMA: results as fp32 units give them.  And operands so small
that their parts end in bf16's subnormals."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from orda_ce_kernel import _native
from oracle.orda_oracle import distillation_loss_oracle
from tests.test_gpu_fp32_precision import _error, _operands
from tests.test_gpu_parity import _make, _np, _orda

pytestmark = pytest.mark.gpu


def _layouts(a, b, splits=1):
    at, bt = a.t().contiguous(), b.t().contiguous()
    yield "K, K", _native.gemm(a, b)
    yield "K, MN", _native.gemm(a, bt, b_mn=True)
    yield "MN, MN", _native.gemm(at, bt, a_mn=True, b_mn=True, splits=splits)


@pytest.mark.parametrize("K", [1, 2, 3, 4, 8, 12, 16])
@pytest.mark.parametrize("kind", ["normal", "positive", "wide"])
def test_short_sums_are_no_less_exact_than_native(kind, K):
    for M, N in ((320, 384), (4096, 2048)):
        a, b = _operands(kind, M, N, K)
        at, bt = (x.t().clone(memory_format=torch.contiguous_format) for x in (a, b))
        pad = -K % 4  # (a K-major operand's rows are read in fours)
        native = _error(_native.gemm(torch.nn.functional.pad(at, (0, 0, 0, pad)),
                                     torch.nn.functional.pad(b, (0, pad)), a_mn=True), a, b)
        got = _error(_native.gemm(at, bt, a_mn=True, b_mn=True), a, b)
        print(f"[short] {kind} K={K} {M}x{N}: {got:.2e}, native {native:.2e}", flush=True)
        assert got <= 1.05 * native


# few outputs (64 x 64 tiles) and many (256 x 128); the infinite values in the
# first, a middle and the last K step and rows, and a tile apart
@pytest.mark.parametrize("M,N,K,splits", [(68, 72, 32, 1), (320, 384, 100, 1), (320, 384, 1000, 3), (4100, 2052, 328, 1)])
def test_infinite_and_huge_operands(M, N, K, splits):
    a, b = _operands("normal", M, N, K)
    cases = [(a, 0, 0, np.inf), (a, M - 1, K - 1, -np.inf), (b, N // 2, K // 2, np.inf), (b, N - 1, 1, -np.inf),
             (a, M // 2, K // 3, 3.4e38), (b, N // 3, K - 2, -3.398e38), (a, 5, 5, np.nan)]
    for x, row, k, value in cases:
        x[row, k] = float(value)
    a[M // 2] *= torch.where(a[M // 2].abs() > 1e38, 1.0, 1e-3)
    b[N // 3] *= torch.where(b[N // 3].abs() > 1e38, 1.0, 1e-3)
    b[:, K // 3] *= 0.01  # (3.4e38 times this stays finite)
    a[:, K - 2] *= 0.01
    exact = a.double() @ b.double().t()
    size = a.double().abs() @ b.double().abs().t()
    fits = size < 3e38  # (beyond, an fp32 sum may overflow in either order)
    for name, c in _layouts(a, b, splits):
        c = c.double()
        assert torch.equal(torch.isnan(c), torch.isnan(exact)), name
        inf = torch.isinf(exact)
        assert torch.equal(c[inf], exact[inf]), name
        err = ((c - exact).abs() / size)[fits & ~torch.isnan(exact)]
        assert float(err.max()) <= (K / 4 + 8) * 2.0 ** -24, (name, float(err.max()))


@pytest.mark.parametrize("M,N", [(320, 384), (4096, 2048)])
@pytest.mark.parametrize("exponent", [-100, -112, -120])
def test_operands_with_parts_in_the_subnormal_range(exponent, M, N):
    """Below 2^-109 the third part is a bf16 subnormal: each product is off by
    2^-133 of the other operand at most, beside a sum's usual rounding."""
    K = 64
    a, b = _operands("normal", M, N, K)
    a = a * 2.0 ** exponent
    exact = a.double() @ b.double().t()
    size = a.double().abs() @ b.double().abs().t()
    bound = b.double().abs().sum(1) * 2.0 ** -133 + (6 * K / 32 + 1) * 2.0 ** -24 * size
    for name, c in _layouts(a, b):
        assert bool(((c.double() - exact).abs() <= bound).all()), name


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("mode,w_t", [("tied", 0.7), ("none", 0.0), ("separate", 0.5)])
@pytest.mark.parametrize("start,length", [(0, 300), (512, 60), (700, 600)])
def test_vocabulary_rows_masked_by_an_infinite_bias(start, length, mode, w_t, train):
    """Hidden states with a constant column and LM heads with the bias there,
    -inf for masked rows: logits of -inf, CE as if the rows were not there."""
    o = _orda()
    N, H, V = 150, 96, 1300
    hs, ht, W, Wt, y = _make(3, N, H, V, torch.float32, w_std=1.5 / H ** 0.5, ignore_frac=0.1)
    hs[:, 7], ht[:, 7] = 1.0, 1.0
    keep = torch.ones(V, dtype=torch.bool)
    keep[start:start + length] = False
    y[(y >= start) & (y < start + length)] = 650
    W[~keep, 7] = -torch.inf
    Wt[~keep, 7] = -torch.inf
    hs_d, W_d = hs.cuda().requires_grad_(train), W.cuda().requires_grad_(True)
    teacher = {"tied": lambda: o.TiedTeacher(ht.cuda()), "separate": lambda: o.SeparateTeacher(ht.cuda(), Wt.cuda()),
               "none": lambda: o.PrecomputedTeacher(logits=torch.zeros(N, V, device="cuda"))}[mode]()
    print(f"[bias] {mode} {start} {length} train={train}", flush=True)
    with torch.set_grad_enabled(train):
        out = o.distillation_loss(hs_d, W_d, y.cuda(), teacher, student_ce_weight=0.8,
                                  teacher_ce_weight=w_t if mode != "none" else None, kl_weight=0.0, backend="hip")
    far = lambda x: torch.where(torch.isinf(x), -300.0, x)  # noqa: E731  (probability 0 in float64 too)
    kw = {"tied": dict(teacher_hidden=_np(ht)), "separate": dict(teacher_hidden=_np(ht), teacher_weight=_np(far(Wt))),
          "none": dict(teacher_logits=np.zeros((N, V)))}[mode]
    ref = distillation_loss_oracle("precomputed" if mode == "none" else mode, _np(hs), _np(far(W)), y.numpy(),
                                   student_ce_weight=0.8, teacher_ce_weight=w_t, kl_weight=0.0, **kw)
    for name in ("loss", "student_ce", "teacher_ce"):
        assert abs(float(getattr(out, name)) - ref[name]) <= 1e-6 + 1e-5 * abs(ref[name]), name
    if train:
        out.loss.backward()
        got, want = _np(W_d.grad), ref["grad_weight"]
        assert np.all(np.isfinite(got))
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
        cols = np.arange(H) != 7  # (the constant column's own gradient is 0 x -inf)
        got, want = _np(hs_d.grad)[:, cols], ref["grad_student_hidden"][:, cols]
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


def test_hidden_rows_past_two_gigabytes_of_a_tile():
    """256 vocabulary rows of 3 x 2^20 fp32 values are 3 GiB: every row counts.
    The products' magnitudes sum to 1.1e3, of which a long fp32 sum is off by
    2.5e-8 and more (2.8e-5 per logit); rows read as zero move the CE by 0.1."""
    o = _orda()
    N, H, V = 5, 3 << 20, 300
    g = torch.Generator(device="cuda").manual_seed(4)
    h = torch.randn(N, H, generator=g, device="cuda")
    W = torch.randn(V, H, generator=g, device="cuda").mul_(H ** -0.5)
    y = torch.tensor([255, 3, 299, 180, 140], device="cuda")
    lt = torch.randn(N, V, generator=g, device="cuda")
    with torch.no_grad():
        out = o.distillation_loss(h, W, y, o.PrecomputedTeacher(logits=lt), kl_weight=0.5, backend="hip")
    x = torch.cat([h.double() @ W[v:v + 50].double().t() for v in range(0, V, 50)], 1)
    logp, logt = torch.log_softmax(x, -1), torch.log_softmax(lt.double(), -1)
    ce = -logp.gather(1, y[:, None]).mean()
    kl = (logt.exp() * (logt - logp)).sum(-1).mean()
    assert abs(float(out.student_ce) - float(ce)) <= 4e-4
    assert abs(float(out.kl) - float(kl)) <= 4e-4
