"""The tile kernel's forms on blocks of 16 x 16: counts of tiles of K around their stages, ragged edges, every epilogue, keys and
values scattered (quads of positions together, quads that start inside one, rows of two sequences in a quad)."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K
import test_tile_forms_gpu as forms
from kernel_helpers import PagedCase

pytestmark = pytest.mark.gpu
BLOCK_FORMS = (2, 3) + tuple(range(6, 15))


@pytest.fixture(autouse=True)
def block_forms(monkeypatch):
    monkeypatch.setitem(forms.FORMS, torch.bfloat16, BLOCK_FORMS)


# (three to eight stages; tiles of 64 to 256 rows and 64 to 256 columns)
@pytest.mark.parametrize("m,n,tiles", [(65, 64, 1), (128, 256, 2), (130, 136, 3), (257, 264, 4), (300, 129, 5), (70, 514, 7), (258, 104, 9), (513, 328, 24)])
def test_epilogues(m, n, tiles):
    forms.test_epilogues_of_every_form(torch.bfloat16, m, n, tiles)


@pytest.mark.parametrize("heads,kv_heads,hd", [(4, 4, 64), (3, 1, 128), (4, 2, 32), (5, 5, 48), (2, 2, 80), (3, 3, 16)])
def test_scattered(heads, kv_heads, hd):
    forms.test_scattered_keys_and_values(torch.bfloat16, heads, kv_heads, hd)


# every activation; no bias, a bias and an output that are not aligned to 16 bytes, rows apart by no whole 16 bytes: whole rows or single values, the same numbers
@pytest.mark.parametrize("m,n", [(130, 328), (257, 104)])
@pytest.mark.parametrize("activation", ["gelu_tanh", "gelu_erf", "squared_relu", None])
def test_activations_and_places(m, n, activation, k=192):
    a, w, bias, want = forms.operands(m, n, k, torch.bfloat16, n)
    function = {"gelu_tanh": lambda x: torch.nn.functional.gelu(x, approximate="tanh"), "gelu_erf": torch.nn.functional.gelu,
                "squared_relu": lambda x: torch.relu(x) ** 2, None: lambda x: x}[activation]
    for form in BLOCK_FORMS:
        shifted = torch.empty(n + 1, device=forms.DEV)[1:]
        shifted.copy_(bias)
        got = {}
        for given in (None, bias.to(forms.DEV), shifted):
            exact = function(want + (bias.double() if given is not None else 0.0))
            for first, pitch in ((0, n), (1, n), (0, n + 3), (4, n + 8)):
                room = torch.full((first + m * pitch + 8,), float("nan"), dtype=torch.bfloat16, device=forms.DEV)
                out = room[first:first + m * pitch].view(m, pitch)[:, :n]
                K.gemm(a.to(forms.DEV), w.to(forms.DEV), K.epilogue_store(out, given) if activation is None else K.epilogue_act(out, activation, given), impl="tile",
                       variant=form)
                # (the output's rounding)
                assert float((out.double().cpu() - exact).abs().max() / exact.abs().max()) < 2.0 ** -8, (form, first, pitch)
                assert int(torch.isnan(room).sum()) == room.numel() - m * n, (form, first, pitch)
                assert torch.equal(out, got.setdefault(given is None, out.clone())), (form, first, pitch)


# the residual stream, sixteen rows at a time: rows and columns that end inside a wave's, beside what is not the product's
@pytest.mark.parametrize("m,n,pitch", [(65, 68, 72), (127, 160, 160), (257, 100, 104), (300, 332, 332), (130, 516, 520)])
def test_residual_stream_between_others(m, n, pitch, k=192):
    a, w, bias, want = forms.operands(m, n, k, torch.bfloat16, m)
    x = torch.randn(m, n, generator=torch.Generator().manual_seed(n))
    for form in BLOCK_FORMS:
        room = torch.full((m + 2, pitch), float("nan"), device=forms.DEV)
        room[:m, :n] = x.to(forms.DEV)
        K.gemm(a.to(forms.DEV), w.to(forms.DEV), K.epilogue_residual(room[:m, :n], bias.to(forms.DEV)), impl="tile", variant=form)
        exact = x.double() + want + bias.double()
        assert float((room[:m, :n].double().cpu() - exact).abs().max() / exact.abs().max()) < 1e-5, form      # (32-bit sums of 192 products and three more)
        assert torch.isnan(room[m:]).all() and torch.isnan(room[:, n:]).all(), form


# tokens of a step in any order: two of every four positions swapped, every fourth position first, two sequences' tokens between each other, drawn
@pytest.mark.parametrize("order", ["swapped", "strided", "between", "drawn"])
def test_scattered_in_any_order(order, heads=3, hd=48, k=128):
    totals = counts = [64, 64, 130, 7]
    width, m = heads * hd, sum(counts)
    if order == "swapped":
        rows = [r ^ 3 if r % 4 in (1, 2) else r for r in range(m - m % 4)] + list(range(m - m % 4, m))
    elif order == "strided":
        rows = [r for first in range(4) for r in range(first, m, 4)]
    elif order == "between":          # a0 b1 b2 a3, b0 a1 a2 b3, ...
        rows = [r + 64 * (r % 4 in (1, 2)) for r in range(64)] + [r + 64 * (r % 4 in (0, 3)) for r in range(64)] + list(range(128, m))
    else:
        rows = torch.randperm(m, generator=torch.Generator().manual_seed(3)).tolist()
    assert sorted(rows) == list(range(m))
    a, w, bias, want = forms.operands(m, 3 * width, k, torch.bfloat16, 5)
    want = want + bias.double()
    for form in BLOCK_FORMS:
        case = PagedCase(totals, counts, heads, hd, torch.bfloat16, forms.DEV, seed=2)
        q = torch.full((m, width), float("nan"), dtype=torch.bfloat16, device=forms.DEV)
        K.gemm(a.to(forms.DEV), w.to(forms.DEV), K.epilogue_qkv(q, width, width, case.view(), case.tok_seq[rows].contiguous(), case.tok_pos[rows].contiguous(),
                                                                bias.to(forms.DEV)), impl="tile", variant=form)
        for got, first in ((case.read_back()[0], width), (case.read_back()[1], 2 * width)):
            error = (got[rows].double().cpu() - want[:, first:first + width]).abs().max() / want.abs().max()
            assert float(error) < 2.0 ** -8, (form, order, first)
