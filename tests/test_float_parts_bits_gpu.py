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
