"""The tile kernel's forms: counts of tiles of K around their stages, ragged edges, every epilogue, keys and values scattered."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K
from kernel_helpers import PagedCase

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FORMS = {torch.bfloat16: (0, 2, 3, 4, 5, 6, 7), torch.float32: (0, 4, 5, 6, 7)}


def operands(m, n, k, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    a, w = torch.randn(m, k, generator=gen).to(dtype), (torch.randn(n, k, generator=gen) * k ** -0.5).to(dtype)
    bias = torch.randn(n, generator=gen)
    return a, w, bias, a.double() @ w.double().t()


# one to seven tiles of K (forms have three to eight stages) and so many that 64 x 64 takes eight, whole and in slices; rows and columns on both sides of whole tiles;
# columns that are no multiple of eight or four, which leave the epilogue's whole rows for single values
@pytest.mark.parametrize("m,n,tiles", [(65, 64, 1), (128, 256, 2), (130, 136, 3), (257, 260, 4), (300, 129, 5), (70, 514, 7),
                                       (70, 130, 49), (130, 200, 150)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_epilogues_of_every_form(dtype, m, n, tiles):
    k = tiles * (64 if dtype == torch.bfloat16 else 32)
    a, w, bias, want = operands(m, n, k, dtype, m + n)
    # float32: sums of k products of size 1 / sqrt(k); bfloat16: the output's rounding
    bound = 1e-5 if dtype == torch.float32 else 2.0 ** -8
    held = torch.full((m, k + 8), float("nan"), dtype=dtype, device=DEV)
    held[:, :k] = a.to(DEV)
    close = lambda got, exact, limit: float((got.double().cpu() - exact).abs().max() / exact.abs().max()) < limit
    for form in FORMS[dtype]:
        room = torch.full((m + 1, n + 8), float("nan"), dtype=dtype, device=DEV)
        for pitch in (n, n + 8):           # rows behind one another, rows apart
            out = room.view(-1)[:m * pitch].view(m, pitch)[:, :n]
            room.fill_(float("nan"))
            K.gemm(held[:, :k], w.to(DEV), K.epilogue_store(out, bias.to(DEV)), impl="tile", variant=form)
            assert close(out, want + bias.double(), bound), (form, pitch, "stored")
            assert torch.isnan(room.view(-1)[m * pitch:]).all() and (pitch == n or torch.isnan(room.view(-1)[:m * pitch].view(m, pitch)[:, n:]).all())
        act = torch.empty(m, n, dtype=dtype, device=DEV)
        K.gemm(held[:, :k], w.to(DEV), K.epilogue_act(act, "gelu_tanh", bias.to(DEV)), impl="tile", variant=form)
        assert close(act, torch.nn.functional.gelu(want + bias.double(), approximate="tanh"), bound), (form, "activated")
        x = torch.randn(m, n)
        stream = x.to(DEV)
        K.gemm(held[:, :k], w.to(DEV), K.epilogue_residual(stream, bias.to(DEV)), impl="tile", variant=form)
        assert close(stream, x.double() + want + bias.double(), 1e-5), (form, "residual")
        parts = torch.full((3, m, n), float("nan"), device=DEV)
        K.gemm(held[:, :k], w.to(DEV), K.epilogue_f32(parts, bias.to(DEV)), impl="tile", variant=form, splits=3)
        assert close(parts.sum(0), want + bias.double(), 1e-5), (form, "slices")


# heads whose columns fill a wave's blocks (64, 128), that leave them (48, 80); sequences that start anywhere in a tile
@pytest.mark.parametrize("heads,kv_heads,hd", [(4, 4, 64), (3, 1, 128), (4, 2, 32), (5, 5, 48), (2, 2, 80)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_scattered_keys_and_values(dtype, heads, kv_heads, hd, k=128):
    totals, counts = [70, 3, 129, 64, 200], [69, 3, 1, 64, 130]
    n_q, n_kv, m = heads * hd, kv_heads * hd, sum(counts)
    a, w, bias, want = operands(m, n_q + 2 * n_kv, k, dtype, hd)
    want = want + bias.double()
    bound = 1e-5 if dtype == torch.float32 else 2.0 ** -8
    for form in FORMS[dtype]:
        case = PagedCase(totals, counts, kv_heads, hd, dtype, DEV, seed=1)
        before_k, before_v = (t.double().cpu() for t in case.read_back())
        q = torch.full((m, n_q), float("nan"), dtype=dtype, device=DEV)
        K.gemm(a.to(DEV), w.to(DEV), K.epilogue_qkv(q, n_q, n_kv, case.view(), case.tok_seq, case.tok_pos, bias.to(DEV)), impl="tile", variant=form)
        after_k, after_v = (t.double().cpu() for t in case.read_back())
        scale = want.abs().max()
        assert float((q.double().cpu() - want[:, :n_q]).abs().max() / scale) < bound, form
        row = at = 0
        for total, count in zip(totals, counts):
            for before, after, first in ((before_k, after_k, n_q), (before_v, after_v, n_q + n_kv)):
                assert torch.equal(after[at:at + total - count], before[at:at + total - count]), form      # older positions stay
                assert float((after[at + total - count:at + total] - want[row:row + count, first:first + n_kv]).abs().max() / scale) < bound, form
            row, at = row + count, at + total


def test_scattered_keys_and_values_behind_a_long_k():
    """The form of 64 x 64 with eight stages among all."""
    test_scattered_keys_and_values(torch.bfloat16, 4, 4, 64, k=49 * 64)
    test_scattered_keys_and_values(torch.bfloat16, 5, 5, 48, k=49 * 64)


def test_which_products_are_the_tile_kernels():
    assert K.own_tiles(610, 3072, 1024, 1024) and K.own_tiles(1024, 2048, 1024, 1024) and K.own_tiles(450, 2048, 4096, 4096)
    assert not K.own_tiles(610, 4096, 1024, 1024) and not K.own_tiles(610, 2048, 4096, 4096)
    assert K.own_tiles(2048, 1600, 1600, 1600, residual=True) and not K.own_tiles(2048, 1600, 1600, 1600)
    assert K.own_tiles(1295, 3072, 1024, 1024, scatters=True) and not K.own_tiles(2048, 3072, 1024, 1024, scatters=True)
    assert not K.own_tiles(2048, 128, 1024, 1024)            # too few tiles
    assert not K.own_tiles(64, 1024, 1024, 1024) and not K.own_tiles(566, 1024, 1000, 1000) and not K.own_tiles(300, 517, 1600, 1600)
    for rows in (65, 256, 257, 384, 512, 513):       # whatever goes by its rows alone stays
        for options in ({}, {"sliced": True}, {"scatters": True}):
            assert K.own_tiles(rows, 4800, 1600, 1600, **options) or not K.deep_form_rows(rows, 1600, 1600, 4800, **options)
