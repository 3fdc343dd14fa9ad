"""Float products of more than 64 rows on tiles brought straight into LDS, against float64."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rel_err(got, want):
    return float((got.detach().cpu().double() - want).abs().max() / want.abs().max())


# edges of tiles of 64 and 128 rows and columns, fewer tiles of K than a form has stages, K no multiple of 32 (the
# general form), slices of K of unequal length, rows that lie apart, sizes on both sides of the rule for the taller tile
@pytest.mark.parametrize("m,n,k,splits", [(65, 40, 32, 1), (128, 64, 64, 1), (129, 65, 96, 2), (200, 130, 36, 1), (300, 517, 416, 3),
                                          (100, 768, 3072, 4), (1000, 2304, 160, 1), (800, 4096, 64, 1)])
@pytest.mark.parametrize("variant", [0, 4, 5, 6, 7])
def test_float_tiles(variant, m, n, k, splits):
    gen = torch.Generator().manual_seed(m + n + k)
    # all 24 bits of the operands count: sums of +-1 nearly cancel and leave their low bits
    a = (1.0 + torch.rand(m, k, generator=gen) * 2.0 ** -12) * torch.where(torch.rand(m, k, generator=gen) < 0.5, -1.0, 1.0)
    w = torch.randn(n, k, generator=gen)
    held = torch.full((m, k + 4), float("nan"), device=DEV)
    held[:, :k] = a.to(DEV)
    want = a.double() @ w.double().t()
    if variant and k % 32:
        with pytest.raises(K.KernelError, match="multiple of 32"):
            K.gemm(held[:, :k], w.to(DEV), K.epilogue_f32(torch.empty(splits, m, n, device=DEV)), impl="tile", variant=variant, splits=splits)
        return
    parts = torch.full((splits, m, n), float("nan"), device=DEV)
    K.gemm(held[:, :k], w.to(DEV), K.epilogue_f32(parts), impl="tile", variant=variant, splits=splits)
    # 32-bit sums of k products of size one: the rounding of a sum of size sqrt(k), k times over, grows as k
    assert rel_err(parts.sum(0), want) < 4e-7 * k ** 0.5 + 2e-6
    if splits == 1:
        bias, out = torch.randn(n, generator=gen), torch.full((m, n), float("nan"), device=DEV)
        K.gemm(held[:, :k], w.to(DEV), K.epilogue_act(out, "gelu_erf", bias.to(DEV)), impl="tile", variant=variant)
        assert rel_err(out, torch.nn.functional.gelu(want + bias.double())) < 4e-7 * k ** 0.5 + 2e-6
        x = torch.randn(m, n, generator=gen)
        stream = x.to(DEV)
        K.gemm(held[:, :k], w.to(DEV), K.epilogue_residual(stream, bias.to(DEV)), impl="tile", variant=variant)
        assert rel_err(stream, x.double() + want + bias.double()) < 4e-7 * k ** 0.5 + 2e-6


def test_slices_of_float_products():
    """As many slices as spread a product's tiles over the compute units, none where they are spread already."""
    assert K.float_split_count(64, 768, 3072) == 1 and K.float_split_count(65, 768, 3070) == 1
    assert K.float_split_count(65, 768, 3072) == 4 and K.float_split_count(256, 768, 768) == 4
    assert K.float_split_count(1200, 768, 3072) == 1 and K.float_split_count(4096, 1600, 1600) == 1
    for rows in (65, 400, 1000, 5000):
        for k in (32, 128, 480, 6400):
            assert 1 <= K.float_split_count(rows, 96, k) <= max(1, min(4, k // 128))
