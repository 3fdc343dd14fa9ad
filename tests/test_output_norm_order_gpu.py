"""The norm of a sublayer's output gives the same numbers however its rows lie in memory."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows that end inside the first and the last quads of both register sizes; partial sums, copies and the next norm's rows apart by
# whole quads or not, and off a quad's start
@pytest.mark.parametrize("width", [8, 1000, 1024, 1028, 2044, 2048])
@pytest.mark.parametrize("kind", ["rms_norm", "layer_norm"])
@pytest.mark.parametrize("parts", [0, 2])
def test_rows_do_not_depend_on_their_places(width, kind, parts):
    gen = torch.Generator().manual_seed(width + parts)
    rows = 7
    rand = lambda *shape: torch.randn(*shape, generator=gen).to(DEV)
    x, gamma, gamma2, bias = rand(rows, width), rand(width), rand(width), rand(width)
    beta = rand(width) if kind == "layer_norm" else None
    held = rand(max(parts, 1), rows, width)

    def run(apart, off):
        place = lambda t: torch.cat([t.new_zeros(off), t.reshape(-1)])[off:].view_as(t)
        delta = held.new_full((held.shape[0], rows, width + apart), float("nan"))
        delta[:, :, :width] = held
        stream = place(x).clone() if off == 0 else place(x)
        cast = torch.full((rows, width + apart), float("nan"), dtype=torch.bfloat16, device=DEV)
        after = torch.full((rows, width + apart), float("nan"), dtype=torch.bfloat16, device=DEV)
        more = {"delta": delta[:, :, :width], "bias": place(bias)} if parts else {"accumulate": False}
        K.output_norm(stream, place(gamma), 1e-5, 0.7, cast=cast[:, :width], kind=kind, beta=beta, then=(kind, gamma2, beta, 1e-5, after[:, :width]), **more)
        return stream, cast[:, :width], after[:, :width]

    want = run(0, 0)
    for apart, off in ((4, 0), (1, 0), (2, 0), (0, 1), (4, 3)):
        for a, b in zip(want, run(apart, off)):
            assert torch.equal(a, b), (apart, off)
