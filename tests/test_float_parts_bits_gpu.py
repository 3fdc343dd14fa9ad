"""Float products made of bfloat16 parts: the bits that the parts leave out, whatever the operands' mantissas."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def product(a, w, variant, splits=1):
    parts = torch.full((splits, a.shape[0], w.shape[0]), float("nan"), device=DEV)
    K.gemm(a.to(DEV), w.to(DEV), K.epilogue_f32(parts), impl="tile", variant=variant, splits=splits)
    return parts.cpu().double().sum(0)


@pytest.mark.parametrize("variant", [6, 7])
def test_products_keep_what_a_rounding_would(variant):
    """What three of the nine products of parts would add is below 2^-24 of the operands' product."""
    gen = torch.Generator().manual_seed(variant)
    # mantissas whose second and third parts are the largest there are (by a search over all 2^23: 0x7fc0, of one sign; cut off
    # instead of rounded, 0x7fff), beside any
    worst = torch.tensor([0x3f807fc0, 0x3f807fff, 0x3f80803f, 0x3f817fff, 0x3fff7fff], dtype=torch.int32)
    any_mantissa = lambda n: torch.randint(0x3f800000, 0x40000000, (n,), generator=gen, dtype=torch.int32)
    x, w = torch.cat([worst, any_mantissa(125)]).view(torch.float32), torch.cat([worst, any_mantissa(195)]).view(torch.float32)
    # every second term takes the leading parts' product away again, so that the sums are small and round where nothing is lost
    turn = lambda v, sign: torch.stack([v, sign * v.to(torch.bfloat16).float()], dim=1).repeat(1, 16)
    a, b = turn(x, -1.0), turn(w, 1.0)
    want = a.double() @ b.double().t()
    # sixteen products, each short of less than 2^-24 of itself; the sums stay below one: a tenth of that for their roundings
    bound = 16 * x.double()[:, None] * w.double()[None, :] * 2.0 ** -24 * 1.1
    assert float(((product(a, b, variant) - want).abs() / bound).max()) < 1.0


@pytest.mark.parametrize("variant", [6, 7])
@pytest.mark.parametrize("m,n,k,splits", [(130, 140, 96, 1), (300, 260, 800, 3)])
def test_tiles_that_are_not_finite_are_the_float_instructions(variant, m, n, k, splits):
    """Where a sum of a tile is not finite the whole tile has the float instructions' numbers, and the other tiles keep theirs."""
    gen = torch.Generator().manual_seed(m + k)
    a, w = torch.randn(m, k, generator=gen), torch.randn(n, k, generator=gen)
    plain, floats = product(a, w, variant, splits), product(a, w, 5, splits)
    for value in (float("nan"), float("inf"), torch.finfo(torch.float32).max):
        held = a.clone()
        held[m - 1, k - 1], held[m - 1, 0] = value, value          # the last block of rows; of slices, the first and the last
        got, want = product(held, w, variant, splits), product(held, w, 5, splits)
        last = (m - 1) // 128 * 128
        assert torch.equal(got[:last], plain[:last])
        assert torch.equal(torch.isnan(got[last:]), torch.isnan(want[last:]))
        if splits == 1:
            assert torch.equal(torch.nan_to_num(got[last:]), torch.nan_to_num(want[last:]))
        else:                # (slices without such a value keep their sums)
            fine = slice(last, m - 1)
            assert float((got[fine] - want[fine]).abs().max() / floats.abs().max()) < 1e-5
        assert torch.equal(got[m - 1], want[m - 1]) or torch.isnan(want[m - 1]).any()


@pytest.mark.parametrize("variant", [6, 7])
@pytest.mark.parametrize("a_exponent,w_exponent", [(-100, 60), (-109, 100), (-118, 100), (-128, 110), (-140, 120), (-70, -58)])
def test_very_small_values(variant, a_exponent, w_exponent):
    """Beside the roundings of any product, a value loses what falls below the smallest bfloat16: 2^-134 at most."""
    gen = torch.Generator().manual_seed(-a_exponent)
    scaled = lambda rows, exponent: (torch.randn(rows, 64, generator=gen, dtype=torch.float64) * 2.0 ** exponent).float()
    a, w = scaled(130, a_exponent), scaled(140, w_exponent)
    want, size = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    lost = 2.0 ** -134 * (w.double().abs().sum(1)[None, :] + a.double().abs().sum(1)[:, None])
    # 24 roundings of a sum of 64 products, each at most 2^-24 of their sizes, what is left out, and sums below the smallest normal float
    bound = 25 * 2.0 ** -24 * size + lost + 64 * 2.0 ** -149
    assert float(((product(a, w, variant) - want).abs() / bound).max()) < 1.0
