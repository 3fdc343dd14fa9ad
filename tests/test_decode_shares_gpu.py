"""Decode attention where only some of a work-group's eight waves have keys: contexts around whole tiles of 32 keys."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K
from kernel_helpers import PagedCase

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("runs", [1, 3, 8])
@pytest.mark.parametrize("q_heads,kv_heads,hd", [(16, 1, 128), (4, 2, 64), (1, 1, 16)])
@pytest.mark.parametrize("window", [0, 40])
def test_decode_of_short_runs(q_heads, kv_heads, hd, runs, window):
    totals = [1, 32, 33, 64, 65, 128, 129, 256, 257, 700]
    n = len(totals)
    case = PagedCase(totals, [1] * n, kv_heads, hd, torch.bfloat16, DEV, seed=4, poison=True)
    gen = torch.Generator().manual_seed(6)
    q = torch.randn(n, q_heads * hd, generator=gen).to(torch.bfloat16).to(DEV)
    out = torch.full((n, q_heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    partial = torch.full((n * q_heads * runs, hd + 2), float("nan"), device=DEV) if runs > 1 else None
    args = K.attention_args(q, out, case.view(), case.tok_seq, case.tok_pos, case.seq_off, case.seq_start, q_heads, n, 1, hd ** -0.5,
                            window, partial)
    K.attention(args, torch.bfloat16, decode=True)
    want = case.reference(q, q_heads, hd ** -0.5, window).double().cpu()
    got = out.double().cpu()
    # weights rounded to bfloat16 before the product with the values (2^-9 of the largest value each) and the output (2^-9)
    assert float((got - want).abs().max() / want.abs().max()) < 2.0 ** -8 + 2.0 ** -9
