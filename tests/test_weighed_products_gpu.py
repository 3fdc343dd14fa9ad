"""The product of experts' units that weighs the experts' sums itself, against float64 and the weights of the kernel that weighs rows."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows on both sides of one a wave, experts and widths whose chunks end in the middle of a batch, a shared expert behind them,
# slices of K that begin inside an expert, both column forms
@pytest.mark.parametrize("rows,experts,top,ff,shared,width", [(1, 8, 2, 64, 0, 64), (8, 8, 2, 96, 32, 200), (9, 3, 3, 32, 256, 48),
                                                              (16, 64, 5, 32, 0, 136), (5, 8, 1, 1024, 1024, 96)])
@pytest.mark.parametrize("score,groups", [("softmax", 1), ("sigmoid", 1), ("chosen", 1)])
@pytest.mark.parametrize("packs", [0, 16, 24])
def test_weighed_sums(rows, experts, top, ff, shared, width, score, groups, packs):
    gen = torch.Generator().manual_seed(rows + ff)
    k = experts * ff + shared
    logits = torch.randn(rows, experts + 4, generator=gen).to(DEV)
    bias, correction = torch.randn(experts, generator=gen).to(DEV), (0.1 * torch.randn(experts, generator=gen)).to(DEV)
    held = torch.randn(rows, k + 8, generator=gen).to(torch.bfloat16).to(DEV)
    w = (torch.randn(width, k, generator=gen) * k ** -0.5).to(torch.bfloat16).to(DEV)
    packed = K.pack_columns(w, packs) if packs else None
    # every token's weights, as the kernel of its own has them: what it makes of ones
    ones = torch.ones(rows, k, device=DEV)
    K.weigh_experts(logits, bias, correction, top, groups, 1, ones, experts, ff, score=score)
    terms = ones.double().cpu() * held[:, :k].double().cpu()
    want, size = terms @ w.double().cpu().t(), terms.abs() @ w.double().cpu().abs().t()
    for splits in (1, 3):
        got = torch.full((splits, rows, width), float("nan"), device=DEV)
        raw = held.clone()
        fits = type("Packed", (), {"for_step": lambda self, m, s: (packed, packs) if packs else None})()
        K.gemm_weighed(logits, bias, correction, top, groups, 1, raw[:, :k], experts, ff, w, K.epilogue_f32(got), splits=splits, packed=fits, score=score)
        assert torch.equal(raw, held)
        # 32-bit sums of k products: at most 2^-24 of their sizes for each
        assert float(((got.sum(0).double().cpu() - want).abs() / (size + 1e-30)).max()) < k * 2.0 ** -24 + 4 * 2.0 ** -24


def test_units_that_are_not_finite_stay_their_users():
    """An expert's units that are infinite or NaN reach the tokens that use it and no other."""
    logits = torch.tensor([[4.0, 0.0, 0.0], [0.0, 4.0, 0.0], [0.0, 0.0, 4.0]], device=DEV)
    hidden = torch.ones(3, 96, dtype=torch.bfloat16, device=DEV)
    hidden[0, 40], hidden[1, 50], hidden[2, 3] = float("inf"), float("nan"), float("-inf")       # (of experts the rows do not use but the second)
    out = torch.empty(1, 3, 16, device=DEV)
    K.gemm_weighed(logits, None, None, 1, 1, 1, hidden, 3, 32, torch.ones(16, 96, dtype=torch.bfloat16, device=DEV), K.epilogue_f32(out))
    assert torch.isnan(out[0, 1]).all() and torch.equal(out[0, 0], torch.full((16,), 32.0, device=DEV)) and torch.equal(out[0, 2], out[0, 0])


def test_refusals():
    logits, w = torch.zeros(17, 8, device=DEV), torch.zeros(16, 256, dtype=torch.bfloat16, device=DEV)
    out = torch.zeros(1, 17, 16, device=DEV)
    with pytest.raises(K.KernelError, match="do not fit"):         # too many rows
        K.gemm_weighed(logits, None, None, 2, 1, 1, torch.zeros(17, 256, dtype=torch.bfloat16, device=DEV), 8, 32, w, K.epilogue_f32(out))
    with pytest.raises(K.KernelError, match="do not fit"):         # chunks of two experts
        K.gemm_weighed(logits, None, None, 2, 1, 1, torch.zeros(8, 256, dtype=torch.bfloat16, device=DEV), 16, 16, w, K.epilogue_f32(out[:, :8]))
