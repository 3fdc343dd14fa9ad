"""The choice of a token's experts, for up to 64 of them, among equal scores, shut-out ones and scores that are no numbers."""
import math

import pytest
import torch

from burn_transformers_amd.kernels import library as K

DEV = "cuda:0"
PATTERNS = 16
pytestmark = pytest.mark.gpu


def chosen_weights(logits, correction, top, groups, keep, score):
    """Best first, the lower index among equals; what ranks at minus infinity or is no number is never chosen."""
    rows, experts = logits.shape
    weights = torch.zeros(rows, experts, dtype=torch.float64)
    for t in range(rows):
        z = [float(v) for v in logits[t].double()]
        if score == "sigmoid":
            s = [1.0 / (1.0 + math.exp(-v)) if v == v else v for v in z]
        else:
            high = max(z)
            s = [math.exp(v - high) for v in z]
            if score == "softmax":
                s = [v / sum(s) for v in s]
        ranked = [(z if score == "chosen" else s)[e] + float(correction[e]) for e in range(experts)]
        if groups > 1:
            per = experts // groups
            best = [max(ranked[g * per:g * per + per]) for g in range(groups)]
            kept = sorted(range(groups), key=lambda g: (-best[g], g))[:keep]
            ranked = [v if e // per in kept else -math.inf for e, v in enumerate(ranked)]
        can = [e for e in range(experts) if ranked[e] > -math.inf]
        picked = sorted(can, key=lambda e: (-ranked[e], e))[:top]
        total = sum(s[e] for e in picked) + 1e-20
        for e in picked:
            weights[t, e] = s[e] / total
    return weights


@pytest.mark.parametrize("score", ["softmax", "sigmoid", "chosen"])
@pytest.mark.parametrize("experts,top,groups,keep", [(1, 1, 1, 1), (8, 2, 1, 1), (9, 2, 3, 2), (8, 2, 4, 2), (16, 1, 1, 1), (17, 1, 1, 1), (31, 31, 1, 1),
                                                     (64, 4, 1, 1), (64, 3, 8, 2), (64, 64, 1, 1), (40, 2, 1, 1)])
def test_ties_and_shut_out_experts(experts, top, groups, keep, score):
    # logits are halves: equal ones are exactly equal, and unequal ones lie far beyond the rounding of a score
    gen = torch.Generator().manual_seed(experts + top)
    logits = torch.randint(-4, 5, (PATTERNS, experts), generator=gen).float() / 2
    correction = torch.zeros(experts)
    if groups == 1 and experts > 2:
        correction[1], correction[experts - 1] = -math.inf, 8.0          # one shut out, one put before all others
        if score == "sigmoid":
            logits[3, 2] = math.nan
    want = chosen_weights(logits, correction, top, groups, keep, score)
    fix = correction.to(DEV)
    units = torch.ones(PATTERNS, experts, device=DEV)
    K.weigh_experts(logits.to(DEV), None, fix, top, groups, keep, units, experts, 1, score=score)
    # every one of 16 columns of the router's rows is one token's logits, exactly
    router = logits.T.contiguous()
    router = torch.nan_to_num(router, nan=-2.0)      # (a product spreads what is no number over all tokens)
    plain = chosen_weights(router.T, correction, top, groups, keep, score)
    found = [(units, want)]
    for tokens in (PATTERNS, 1800) if experts <= 31 else (PATTERNS,):
        at = torch.arange(tokens) % PATTERNS
        weights = torch.full((tokens, experts), math.nan, device=DEV)
        K.route(torch.eye(PATTERNS)[at].to(DEV), router.to(DEV), fix, top, groups, keep, weights, score=score)
        found.append((weights, plain[at]))
    for got, expected in found:
        got = got.cpu().double()
        assert torch.equal(got != 0, expected != 0), "another expert was chosen"
        # an exponential, a sum of 64 and two divisions in 32 bits
        assert float((got - expected).abs().max()) < 80 * 2.0 ** -24


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
# (the two kernels add a logit's products in different orders: steps below the line have the sums of a work-group a token, bit for bit)
@pytest.mark.parametrize("outputs,width,below,above", [(9, 1024, [1279, 1280, 1535], 1536), (17, 1024, [1280, 1535], 1536), (8, 512, [1280, 1535], 1536),
                                                       (8, 1024, [1536, 1791], 1792)])
def test_sums_on_both_sides_of_the_line(outputs, width, below, above, dtype):
    gen = torch.Generator().manual_seed(outputs)
    h = torch.randn(above, width, generator=gen).to(getattr(torch, dtype)).to(DEV)
    router = (torch.randn(outputs, width, generator=gen) * width ** -0.5).to(DEV)

    def weights(rows):
        out = torch.full((rows.shape[0], outputs), math.nan, device=DEV)
        K.route(rows, router, None, outputs, 1, 1, out, score="softmax")          # (all are chosen: their scores as they are)
        return out
    few = torch.cat([weights(h[begin:begin + 100]) for begin in range(0, above, 100)])
    for tokens in below:
        assert torch.equal(weights(h[:tokens]), few[:tokens]), tokens
    # sums of `width` products of size one in another order
    many = weights(h)
    assert not torch.equal(many, few) and float((many - few).abs().max()) < 4e-6
