"""The skinny product where an offset inside its rows, or inside a work-group's columns, takes more than 31 bits: rows of a view 2 GiB apart
and a K of many millions, with every epilogue, packed weights and chunk-major rows."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from burn_transformers_amd.kernels import library as K  # noqa: E402
from kernel_helpers import PagedCase  # noqa: E402
from test_skinny_forms_gpu import DEV, in_chunks  # noqa: E402


@pytest.mark.parametrize("rows,apart", [(3, 2 ** 31 + 64), (33, 2 ** 26 + 64)])        # (the third row starts beyond 4 GiB)
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("columns", [8, 28])
def test_rows_far_apart(rows, apart, dtype, columns):
    dt, k, hd = getattr(torch, dtype), 1096, 48
    n, size = 4 * hd, 2 if dtype == "bfloat16" else 4
    gen = torch.Generator().manual_seed(rows)
    near = torch.randn(rows, k, generator=gen).to(dt).to(DEV)
    base = torch.empty((rows - 1) * apart // size + k, dtype=dt, device=DEV)
    far = base.as_strided((rows, k), (apart // size, 1)).copy_(near)
    w = (torch.randn(n, k, generator=gen) * k ** -0.5).to(dt).to(DEV)
    bias = torch.randn(n, generator=gen).to(DEV)
    frequencies = torch.rand(10, generator=gen).to(DEV)
    residual = torch.randn(rows, n, generator=gen).to(DEV)
    case = PagedCase([1 + (37 * i) % 200 for i in range(rows)], [1] * rows, 1, hd, dt, DEV, seed=rows)

    def products(a):
        def new(*shape, dtype=dt):
            return torch.full(shape, float("nan"), dtype=dtype, device=DEV)
        outs = [new(2, rows, n, dtype=torch.float32), new(rows, n), residual.clone(), new(rows, 2 * hd), new(rows, 180),
                new(rows, 100, dtype=torch.float32), new(rows, n - 100)]
        case.keys.fill_(float("nan"))
        case.values.fill_(float("nan"))
        for epilogue, weights, splits in [(K.epilogue_f32(outs[0], bias), w, 2), (K.epilogue_act(outs[1], "gelu_tanh", bias), w, 1),
                                          (K.epilogue_residual(outs[2], bias), w, 1),
                                          (K.epilogue_qkv(outs[3], 2 * hd, hd, case.view(), case.tok_seq, case.tok_pos, bias), w, 1),
                                          (K.epilogue_turn(outs[4], 36, 4, 20, frequencies, case.tok_pos, 1.25), w[:180], 1),
                                          (K.epilogue_f32_act(outs[5], 100, outs[6], "squared_relu"), w, 1)]:
            K.gemm(a, weights, epilogue, splits=splits, impl="skinny", variant=columns)
        ends = (torch.tensor(case.totals).cumsum(0) - 1).to(DEV)
        assert not any(bool(out.isnan().any()) for out in outs)
        return outs + [t[ends.to(t.device)] for t in case.read_back()]
    # (rows side by side take another form of the kernel with the same sums)
    assert all(torch.equal(f, s) for f, s in zip(products(far), products(near)))


@pytest.mark.parametrize("packed", [False, True])
def test_many_millions_of_columns(packed):
    # 32 columns of the weights are more than 2 GiB; zeros but for places at both ends of K, of its last whole chunk and in between
    k, n, rows = 2 ** 25 + 40, 32, 3
    gen = torch.Generator().manual_seed(7)
    places = torch.tensor([0, 31, 2 ** 24 + 3, 2 ** 25 - 1, 2 ** 25 + 31, 2 ** 25 + 32, k - 1])
    some, those = torch.randn(rows, len(places), generator=gen).bfloat16(), torch.randn(n, len(places), generator=gen).bfloat16()
    a, w = (torch.zeros(count, k, dtype=torch.bfloat16, device=DEV) for count in (rows, n))
    a[:, places.to(DEV)], w[:, places.to(DEV)] = some.to(DEV), those.to(DEV)
    out = torch.full((1, rows, n), float("nan"), device=DEV)
    K.gemm(a, w, K.epilogue_f32(out, None), impl="skinny", variant=32, **({"packed": (K.pack_columns(w, 32), 32)} if packed else {}))
    exact, size = some.double() @ those.double().T, some.double().abs() @ those.double().abs().T
    assert bool(((out[0].cpu().double() - exact).abs() <= 8 * 2.0 ** -24 * size).all())        # seven products and their sums


def test_chunks_of_many_rows():
    k, n, rows = 2 ** 24 + 32, 8, 64
    gen = torch.Generator().manual_seed(8)
    places = torch.tensor([0, 31, 2 ** 23 + 3, 2 ** 24 - 1, k - 1])
    some, those = torch.randn(rows, len(places), generator=gen).bfloat16(), torch.randn(n, len(places), generator=gen).bfloat16()
    a, w = (torch.zeros(count, k, dtype=torch.bfloat16, device=DEV) for count in (rows, n))
    a[:, places.to(DEV)], w[:, places.to(DEV)] = some.to(DEV), those.to(DEV)
    sums, activated = torch.full((rows, 4), float("nan"), device=DEV), torch.full((rows, 4), float("nan"), dtype=torch.bfloat16, device=DEV)
    K.gemm(in_chunks(a), w, K.epilogue_f32_act(sums, 4, activated, "squared_relu"), impl="skinny")
    exact, size = some.double() @ those.double().T, some.double().abs() @ those.double().abs().T
    assert bool(((sums.cpu().double() - exact[:, :4]).abs() <= 6 * 2.0 ** -24 * size[:, :4]).all())
    want = exact[:, 4:].clamp_min(0).square()
    assert bool(((activated.cpu().double() - want).abs() <= 2.0 ** -8 * want + 16 * 2.0 ** -24 * size[:, 4:].square()).all())
