"""The skinny product's forms for few rows, which load several chunks of K together: every form against float64, and bit for bit
the rows that the form for sixteen rows gives (only the lanes that hold a value differ, never the order of a sum).  The epilogues that look
something up in the step's tables, in every form: against what the plainest epilogue leaves of the same sums."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from burn_transformers_amd.kernels import library as K  # noqa: E402
from kernel_helpers import PagedCase, gelu_tanh  # noqa: E402

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


def sums_of(a, w, columns, rows, bias=None):
    """The product's sums in 32 bits, by the same form with the plainest epilogue."""
    out = torch.full((1, rows, w.shape[0]), float("nan"), device=DEV)
    K.gemm(a, w, K.epilogue_f32(out, bias), impl="skinny", variant=columns)
    return out[0]


def in_chunks(a):
    """The same rows chunk-major, with columns of zeros behind the last."""
    rows, columns = a.shape
    chunk = 64 // a.element_size()
    padded = torch.nn.functional.pad(a, (0, -columns % chunk))
    return K.Chunked(padded.view(rows, -1, chunk).permute(1, 0, 2).contiguous().view(rows, -1), rows, columns)


# rows on both sides of every form, chunks a wave on both sides of the longest batch, widths that leave a last work-group part of its columns
@pytest.mark.parametrize("chunks,extra", [(9, 0), (33, 8), (64, 0), (75, 8)])
@pytest.mark.parametrize("columns", [8, 12, 16, 28])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_epilogues_with_tables(chunks, extra, columns, dtype):
    dt = getattr(torch, dtype)
    k = chunks * (32 if dtype == "bfloat16" else 16) + extra
    gen = torch.Generator().manual_seed(chunks + columns)
    hd, pitch, at, dim = 48, 36, 4, 20
    n = 4 * hd                                 # two heads of queries on one of keys and values; turned: 180 columns
    w = (torch.randn(n, k, generator=gen) / math.sqrt(k)).to(dt).to(DEV)
    bias = torch.randn(n, generator=gen).to(DEV)
    frequencies = (100.0 ** (-torch.arange(dim // 2, dtype=torch.float64) * 2 / dim)).float().to(DEV)
    for m in (1, 4, 5, 8, 9, 16, 17, 32, 33, 64):
        rows = torch.randn(m, k, generator=gen)
        kinds = [rows.to(dt).to(DEV)]
        if dtype == "bfloat16" and m <= 16 and k <= 2048 and k % 8 == 0:
            kinds.append(K.Normalized(rows.to(DEV), torch.ones(k, device=DEV), None, 1e-5, "rms_norm"))
        for a in kinds:
            # into the cache, at positions in and at the ends of blocks
            case = PagedCase([1 + (37 * i) % 200 for i in range(m)], [1] * m, 1, hd, dt, DEV, seed=m)
            q = torch.full((m, 2 * hd), float("nan"), dtype=dt, device=DEV)
            K.gemm(a, w, K.epilogue_qkv(q, 2 * hd, hd, case.view(), case.tok_seq, case.tok_pos, bias), impl="skinny", variant=columns)
            want = sums_of(a, w, columns, m, bias).to(dt)
            ends = torch.tensor(case.totals).cumsum(0) - 1
            keys, values = (t[ends.to(DEV)] for t in case.read_back())
            assert torch.equal(torch.cat([q, keys, values], 1), want), m
            # turned: the sums in 32 bits, an angle in 32 bits, its sine and cosine, a product and a sum
            turned = torch.full((m, 180), float("nan"), dtype=dt, device=DEV)
            places = (case.tok_pos + 300).contiguous()
            K.gemm(a, w[:180], K.epilogue_turn(turned, pitch, at, dim, frequencies, places, 1.25), impl="skinny", variant=columns)
            v = sums_of(a, w[:180], columns, m).cpu().double().view(m, -1, pitch)
            angle = (places.float()[:, None] * frequencies).cpu().double()[:, None]
            part = v[..., at:at + dim].unflatten(-1, (-1, 2))
            one, two, cs, sn = part[..., 0], part[..., 1], 1.25 * torch.cos(angle), 1.25 * torch.sin(angle)
            exact = v.clone()
            exact[..., at:at + dim] = torch.stack([one * cs - two * sn, two * cs + one * sn], -1).flatten(-2)
            size = v.abs().clone()
            size[..., at:at + dim] = 1.25 * (one.abs() + two.abs()).repeat_interleave(2, -1)
            error = (turned.cpu().double().view(m, -1, pitch) - exact).abs()
            last = 2.0 ** -8 if dtype == "bfloat16" else 0.0              # (half a unit of eight bits)
            assert bool((error <= 8 * 2.0 ** -24 * size + last * exact.abs() * 1.01).all()), m
            # some columns in 32 bits, the others activated; rows row-major or in chunks
            for chunked in (False, True) if not isinstance(a, K.Normalized) and m <= K.Chunked.MAX_ROWS else (False,):
                sums, activated = torch.full((m, 100), float("nan"), device=DEV), torch.full((m, n - 100), float("nan"), dtype=dt, device=DEV)
                given = in_chunks(a) if chunked else a
                K.gemm(given, w, K.epilogue_f32_act(sums, 100, activated, "squared_relu"), impl="skinny", variant=columns)
                want = sums_of(a, w, columns, m)
                assert torch.equal(sums, want[:, :100]) and torch.equal(activated, want[:, 100:].clamp_min(0).square().to(dt)), (m, chunked)
