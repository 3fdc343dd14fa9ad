"""Float products made of bfloat16 parts: their error beside the float instructions', and values that have no parts."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def product(a, w, variant, splits=1):
    parts = torch.full((splits, a.shape[0], w.shape[0]), float("nan"), device=DEV)
    K.gemm(a.to(DEV), w.to(DEV), K.epilogue_f32(parts), impl="tile", variant=variant, splits=splits)
    return parts.cpu().double().sum(0)


# one tile of K and each count around the two that are on their way, edges of tiles, slices; variant 0 reaches 6 and 7 by its rule
@pytest.mark.parametrize("m,n,k,splits", [(1, 1, 32, 1), (129, 127, 64, 1), (127, 129, 96, 1), (130, 260, 128, 3), (257, 70, 800, 1),
                                          (700, 2304, 768, 1), (1100, 3072, 768, 1)])
@pytest.mark.parametrize("variant", [0, 6, 7])
def test_error_is_no_larger_than_the_float_instructions(variant, m, n, k, splits):
    gen = torch.Generator().manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=gen), torch.randn(n, k, generator=gen) * 0.02
    want = a.double() @ w.double().t()
    size = a.double().abs() @ w.double().abs().t()
    error = lambda got: float((got - want).norm() / size.norm())
    # a handful of sums may round either way: one rounding of a sum of the products' sizes, 2^-24, beside the other form's error
    slack = 2.0 ** -24 if m * n < 100 else 0.0
    assert error(product(a, w, variant, splits)) <= error(product(a, w, 5, splits)) + slack


@pytest.mark.parametrize("variant", [6, 7])
def test_values_without_parts(variant):
    """Infinities, NaN and floats beyond the largest bfloat16 give what the float instructions give, in their places only."""
    gen = torch.Generator().manual_seed(7)
    a, w = torch.randn(200, 160, generator=gen), torch.randn(150, 160, generator=gen)
    a[3, 5], a[70, 159], a[131, 0], a[199, 64] = float("inf"), float("nan"), torch.finfo(torch.float32).max, -float("inf")
    w[:, 0] = 0.25
    w[9, 5] = 0.0
    w[149, 100] = float("inf")
    w[7] = w[8].sign()                     # values with one part only
    want, got = product(a, w, 1), product(a, w, variant)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf], want[inf])
    fine = torch.isfinite(want)
    assert int((~fine).sum()) >= 4 * 150 - 160 and float(want[131, 1]) > 5e37
    exact = a.double() @ w.double().t()
    size = a.double().abs() @ w.double().abs().t()
    # 160 products: each sum's rounding is at most 2^-24 of the sum of the products' sizes
    assert float(((got - exact).abs() / size)[fine].max()) < 160 * 2.0 ** -24
