"""The sums of a norm on both sides of the rule that chooses the rotation's kernel: the two kernels add a norm's squares in different
orders, so a step's tokens have the sums of the kernel that the rule names, bit for bit, however many tokens are beside them."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K
from kernel_helpers import PagedCase

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rotated(tokens, heads, kv_heads, dim, whole):
    """(queries, keys) of the first ``tokens`` of one sequence, whose values do not depend on how many are taken."""
    case = PagedCase([tokens], [tokens], kv_heads, dim, torch.float32, DEV, seed=1)
    gen = torch.Generator().manual_seed(heads)
    fused = torch.randn(1600, (heads + 2 * kv_heads) * dim, generator=gen)[:tokens].to(DEV)
    gammas = [torch.randn((n if whole else 1) * dim, generator=gen).to(DEV) for n in (heads, kv_heads)]
    q_out = torch.full((tokens, heads * dim), float("nan"), device=DEV)
    frequencies = (1000.0 ** (-2.0 * torch.arange(16) / 32)).to(DEV)
    K.head_rotary(fused, heads, kv_heads, dim, dim, 32, frequencies, *gammas, 1e-3, q_out, case.tok_seq, case.tok_pos, case.view(), torch.float32,
                  whole_norm=whole)
    return q_out.cpu(), case.read_back()[0]


@pytest.mark.parametrize("heads,kv_heads,dim,whole,many,few", [
    (8, 2, 128, True, [128, 129, 300, 511, 512, 1100], []),           # 1,024 channels under one norm: from 128 tokens on
    (16, 4, 128, True, [128, 200, 255, 256], []),
    (6, 2, 128, True, [615, 768], [512, 613]),                        # fewer: from 6,144 heads of all tokens on
    (3, 1, 128, False, [1536, 1600], [1229, 1300, 1535]),             # a norm a head: from 7,680
])
def test_sums_of_a_norm_by_the_rule(heads, kv_heads, dim, whole, many, few):
    above, below = rotated(1600, heads, kv_heads, dim, whole), rotated(100, heads, kv_heads, dim, whole)
    assert not torch.equal(above[0][:100], below[0]), "the kernels' sums differ, or this test says nothing"
    for tokens in many:
        got = rotated(tokens, heads, kv_heads, dim, whole)
        assert all(torch.equal(g, w[:tokens]) for g, w in zip(got, above)), tokens
    for tokens in few:
        got = rotated(tokens, heads, kv_heads, dim, whole)
        assert all(torch.equal(g[:100], w) for g, w in zip(got, below)), tokens
