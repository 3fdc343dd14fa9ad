"""The norm of a sublayer's output at widths and pitches on both sides of what is read four columns at a time, against float64."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one quad or one column of the last thread, a row that ends inside the block, both register sizes, rows of the partial sums
# and of the copies that are and are not whole quads apart
@pytest.mark.parametrize("width", [4, 1000, 1022, 1024, 1028, 2044, 2046, 2048])
@pytest.mark.parametrize("pad", [0, 2, 4])
@pytest.mark.parametrize("kind", ["rms_norm", "layer_norm"])
@pytest.mark.parametrize("parts", [1, 5])
def test_rows(width, pad, kind, parts):
    gen = torch.Generator().manual_seed(width + parts)
    rows = 3
    rand = lambda *shape: torch.randn(*shape, generator=gen)
    x, gamma, beta, gamma2, bias = rand(rows, width), rand(width), rand(width), rand(width), rand(width)
    held = torch.full((parts, rows, width + pad), float("nan"))
    held[:, :, :width] = rand(parts, rows, width)
    beta = beta if kind == "layer_norm" else None

    def norm(v, gamma, beta, eps):
        v = v - v.mean(1, keepdim=True) if kind == "layer_norm" else v
        v = v / torch.sqrt((v * v).mean(1, keepdim=True) + eps) * gamma.double()
        return v + beta.double() if beta is not None else v
    want = x.double() + 0.7 * norm(held[:, :, :width].double().sum(0) + bias.double(), gamma, beta, 1e-4)
    stream = x.to(DEV)
    cast = torch.full((rows, width + 2 + pad), float("nan"), dtype=torch.bfloat16, device=DEV)
    after = torch.full((rows, width + pad), float("nan"), dtype=torch.bfloat16, device=DEV)
    move = lambda t: t.to(DEV) if t is not None else None
    K.output_norm(stream, gamma.to(DEV), 1e-4, 0.7, delta=held.to(DEV)[:, :, :width], bias=bias.to(DEV), cast=cast, kind=kind, beta=move(beta),
                  then=(kind, gamma2.to(DEV), move(beta), 1e-5, after[:, :width]))
    close = lambda got, exact, limit: float((got.double().cpu() - exact).abs().max() / exact.abs().max()) < limit
    assert close(stream, want, 1e-5)                                   # 32-bit sums over a row
    assert close(cast[:, :width], want, 2.0 ** -8) and float(cast[:, width:].abs().max()) == 0.0
    assert close(after[:, :width], norm(want, gamma2, beta, 1e-5), 2.0 ** -8) and (pad == 0 or torch.isnan(after[:, width:]).all())
