"""Decode attention over block tables around 64 entries (a lane of a wave holds one entry each; later ones are looked up): with and
without a window, in one run and in several, with more query heads than fill a work-group once and a gate and a sink."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from burn_transformers_amd.kernels import library as K  # noqa: E402
from kernel_helpers import PagedCase  # noqa: E402
from test_kernels_gpu import DEV, rel_err  # noqa: E402
from test_rotutar_kernels_gpu import sink_reference  # noqa: E402


@pytest.mark.parametrize("window", [0, 300])
@pytest.mark.parametrize("runs", [1, 3, 11])             # (the kernels that join read eight records at a time)
@pytest.mark.parametrize("hd,dtype", [(64, "bfloat16"), (128, "bfloat16"), (16, "float32"), (64, "float32"), (80, "float32"), (128, "float32")])
@pytest.mark.parametrize("totals", [[1, 513, 30], [4095, 4096, 4097, 4161], [5000, 12, 8190]])
def test_tables_around_a_wave(totals, hd, dtype, runs, window):
    dt = getattr(torch, dtype)
    case = PagedCase(totals, [1] * len(totals), 2, hd, dt, DEV, seed=hd + len(totals))
    gen = torch.Generator().manual_seed(hd)
    q = (torch.randn(len(totals), 8 * hd, generator=gen) * 0.5).to(dt).to(DEV)
    out = torch.full((len(totals), 8 * hd), float("nan"), dtype=dt, device=DEV)
    partial = torch.full((len(totals) * 8 * runs, hd + 2), float("nan"), device=DEV) if runs > 1 else None
    args = K.attention_args(q, out, case.view(), case.tok_seq, case.tok_pos, case.seq_off, case.seq_start,
                            8, len(totals), 1, 0.3, window, partial)
    K.attention(args, dt, decode=True)
    # bfloat16: probabilities and stored rows, 2^-9 each, relative to the largest value of a row of weights of one; float32: sums
    # of products, their exponentials and a sum over the keys, some twenty roundings each
    assert rel_err(out, case.reference(q, 8, 0.3, window)) < (1.2e-2 if dtype == "bfloat16" else 40 * 2.0 ** -24)


# one head a work-group, more elements than threads; runs: whole, and around the eight records that a join reads together
@pytest.mark.parametrize("runs", [1, 3, 11])
@pytest.mark.parametrize("heads,kv", [(4, 4), (16, 1)])
@pytest.mark.parametrize("span", [0, 1])
@pytest.mark.parametrize("hd,dtype", [(128, "bfloat16"), (128, "float32"), (64, "float32")])
def test_gates_and_sinks_asked_for_early(runs, heads, kv, span, hd, dtype):
    dt, totals = getattr(torch, dtype), [700, 65, 1]
    case = PagedCase(totals, [1] * 3, kv, hd, dt, DEV, seed=heads)
    gen = torch.Generator().manual_seed(heads + span)
    q = (torch.randn(3, heads * hd, generator=gen) * 0.5).to(dt).to(DEV)
    sink = torch.randn(heads, generator=gen) + torch.arange(heads) % 2 * 6           # (up to the size of all keys together)
    gate = torch.randn(3, heads * (hd - 16 if span else 1), generator=gen).to(DEV)
    partial = torch.full((3 * heads * runs, hd + 2), float("nan"), device=DEV) if runs > 1 else None

    def attend(**more):
        out = torch.full((3, heads * hd), float("nan"), dtype=torch.float32 if "gate" in more else dt, device=DEV)
        args = K.attention_args(q, out, case.view(), case.tok_seq, case.tok_pos, case.seq_off, case.seq_start, heads, 3, 1, 0.3, 0, partial,
                                sink=sink.to(DEV), **more)
        K.attention(args, dt, decode=True)
        return out.cpu().double().view(3, heads, hd)
    plain = attend()
    # (the bounds of the test above, of every sequence's and head's row: a short context's rows are its values' size)
    exact = sink_reference(case, q, heads, 0.3, 0, sink).view(3, heads, hd)
    row_error = (plain - exact).norm(dim=-1) / exact.norm(dim=-1)
    assert float(row_error.max()) < (1.2e-2 if dtype == "bfloat16" else 40 * 2.0 ** -24)
    other = sink_reference(case, q, heads, 0.3, 0, sink.roll(1)).view(3, heads, hd)
    assert bool(((other - exact).norm(dim=-1) / exact.norm(dim=-1)).gt(0.1).sum(1).ge(heads // 4).all()), "another head's sink would not show"
    factor = torch.sigmoid(gate.cpu().double()).view(3, heads, -1)
    if span:
        factor = torch.cat([factor, torch.ones(3, heads, 16, dtype=torch.float64)], -1)
    gated = attend(gate=gate, gate_dim=hd - 16 if span else 0)
    last = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -20        # the rounding of the row without a gate, or the sigmoid's
    assert bool(((gated - plain * factor).abs() <= last * plain.abs() + 1e-6).all())
