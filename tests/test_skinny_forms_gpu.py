"""The skinny product's forms for few rows, which load several chunks of K together: every form against float64, and bit for bit
the rows that the form for sixteen rows gives (only the lanes that hold a value differ, never the order of a sum)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from burn_transformers_amd.kernels import library as K  # noqa: E402
from kernel_helpers import gelu_tanh  # noqa: E402

DEV = "cuda:0"


# one chunk a wave, loads of several chunks with the last ones missing, a second batch, a partial chunk behind each
@pytest.mark.parametrize("chunks", [8, 33, 43, 64, 75, 130])
@pytest.mark.parametrize("extra", [0, 8])
@pytest.mark.parametrize("columns", [8, 12, 16, 28])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_few_rows_are_the_rows_of_sixteen(chunks, extra, columns, dtype):
    dt = getattr(torch, dtype)
    k, n = chunks * (32 if dtype == "bfloat16" else 16) + extra, 90
    gen = torch.Generator().manual_seed(chunks + columns)
    a = torch.randn(16, k, generator=gen).to(dt).to(DEV)
    w = (torch.randn(n, k, generator=gen) / math.sqrt(k)).to(dt).to(DEV)
    bias = torch.randn(n, generator=gen).to(DEV)
    exact = a.cpu().double() @ w.cpu().double().t()
    # a sum of k products, rounded once per instruction of at least four of them and once per wave
    bound = (k / 4 + 8) * 2.0 ** -24 * (a.cpu().double().abs() @ w.cpu().double().abs().t()) + 1e-30
    packed = (K.pack_columns(w, columns), columns)
    for splits in (1, 2):
        whole = torch.full((splits, 16, n), float("nan"), device=DEV)
        K.gemm(a, w, K.epilogue_f32(whole), splits=splits, impl="skinny", variant=columns)
        assert bool(((whole.sum(0).cpu().double() - exact).abs() <= 2 * bound).all())
        for m in (1, 4, 5, 8, 9):
            for given in (None, packed):
                few = torch.full((splits, m, n), float("nan"), device=DEV)
                K.gemm(a[:m], w, K.epilogue_f32(few), splits=splits, impl="skinny", variant=0 if given else columns, packed=given)
                assert torch.equal(few, whole[:, :m]), (m, splits, given is not None)
    for m in (1, 4, 8, 16):                   # into the stream, and activated
        stream = torch.randn(m, n, generator=gen).to(DEV)
        want = stream.cpu().double() + exact[:m] + bias.cpu().double()
        K.gemm(a[:m], w, K.epilogue_residual(stream, bias), impl="skinny", variant=columns)
        assert bool(((stream.cpu().double() - want).abs() <= bound[:m] + 2.0 ** -22 * (want.abs() + 4)).all())
        out = torch.full((m, n), float("nan"), dtype=dt, device=DEV)
        K.gemm(a[:m], w, K.epilogue_act(out, "gelu_tanh", bias), impl="skinny", variant=columns)
        want = gelu_tanh(exact[:m] + bias.cpu().double())
        last = 2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -20        # of the stored type; the GELU's slope is below 1.13
        assert bool(((out.cpu().double() - want).abs() <= 1.13 * bound[:m] + last * want.abs() + 2.0 ** -20).all())
