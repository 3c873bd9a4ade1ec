"""The split-operand fp32 GEMM against float64, beside the native fp32 MFMA
kernel on the same operands (orda_gemm keeps that for an MN-major A with a
K-major B).  Sums of 64 products and more are no less exact than native ones:
the errors are means over 10^5 and more outputs, which repeat to a few per
cent, so 1.05 of the native error is allowed."""
from __future__ import annotations

import pytest
import torch

from orda_ce_kernel import _native

pytestmark = pytest.mark.gpu


def _operands(kind, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randn(n, K, generator=g, device="cuda") for n in (M, N))
    if kind == "positive":
        a, b = a.abs(), b.abs()
    elif kind == "wide":  # magnitudes over ten orders: probabilities
        a, b = torch.exp(4 * a), torch.exp(4 * b)
    elif kind == "mixed":
        a = torch.exp(4 * a)
    return a, b


def _error(c, a, b):
    """Root mean square error relative to the sum of the products' magnitudes."""
    exact = a.double() @ b.double().t()
    size = a.double().abs() @ b.double().abs().t()
    return float(((c.double() - exact) / size).pow(2).mean().sqrt())


# 64 x 64 and 256 x 128 tiles (few and many outputs)
@pytest.mark.parametrize("M,N", [(320, 384), (4096, 2048)])
@pytest.mark.parametrize("K", [64, 200, 1024, 4096])
@pytest.mark.parametrize("kind", ["normal", "positive", "wide", "mixed"])
def test_long_sums_are_no_less_exact_than_native(kind, K, M, N):
    a, b = _operands(kind, M, N, K)
    at, bt = a.t().contiguous(), b.t().contiguous()
    native = _error(_native.gemm(at, b, a_mn=True), a, b)
    for name, c in (("K, K", _native.gemm(a, b)), ("K, MN", _native.gemm(a, bt, b_mn=True)),
                    ("MN, MN", _native.gemm(at, bt, a_mn=True, b_mn=True))):
        got = _error(c, a, b)
        print(f"[precision] {kind} K={K} {M}x{N} {name}: {got:.2e}, native {native:.2e}", flush=True)
        assert got <= 1.05 * native, name


def test_dropped_products_of_the_worst_operands():
    """0x3f80ff80: all bits below the first part's at their largest.  One
    product of four, the rest zero: within the dropped 2^-24 and one rounding."""
    x = torch.tensor(0x3f80ff80, dtype=torch.int32).view(torch.float32).item()
    a, b = torch.zeros(64, 4, device="cuda"), torch.zeros(64, 4, device="cuda")
    a[:, 1] = x
    b[:, 1] = x
    c = _native.gemm(a, b)
    assert float((c.double() - x * x).abs().max()) <= 2.0 ** -23 * x * x
