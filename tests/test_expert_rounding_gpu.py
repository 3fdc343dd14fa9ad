"""Where the units of a step's experts are rounded: a token's results are the same numbers in small steps as in larger ones."""

import pytest
import torch

from burn_transformers_amd.parts.experts import RoutedExperts
from step_helpers import make_step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one row to the most the skinny kernel takes, on both sides of its blocks of sixteen
@pytest.mark.parametrize("rows", [1, 8, 16, 17, 40])
@pytest.mark.parametrize("shared_ff", [0, 96])
@pytest.mark.parametrize("unit,score", [("squared_relu", "chosen"), ("gelu_erf", "sigmoid")])
def test_units_are_rounded_once_weighed(rows, shared_ff, unit, score):
    """Units come out of the first product in bfloat16, are weighed in 32-bit and rounded to bfloat16 again, whatever the step's size."""
    experts, top, ff, width = 8, 2, 64, 128
    gen = torch.Generator().manual_seed(rows + shared_ff)
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16)
    held = {"router": draw(experts, width).float()}
    for name, wide in [(str(e), ff) for e in range(experts)] + ([("shared", shared_ff)] if shared_ff else []):
        held["up_" + name if name != "shared" else "shared_up"] = draw(wide, width)
        held["down_" + name if name != "shared" else "shared_down"] = draw(width, wide)
    params = {"width": width, "experts": experts, "top": top, "ff": ff, "shared_ff": shared_ff, "unit": unit, "score": score, "normalize": True}
    part = RoutedExperts(params, {k: v.to(DEV) for k, v in held.items()})
    h = (0.1 * torch.randn(rows, width, generator=gen)).to(torch.bfloat16)
    got = part.forward(h.to(DEV), make_step(torch.bfloat16, [rows]), None).partials.double().sum(0).cpu()

    x, rounded = h.double(), lambda t: t.to(torch.bfloat16).double()
    act = (lambda v: torch.relu(v) ** 2) if unit == "squared_relu" else torch.nn.functional.gelu
    logits = x @ held["router"].double().t()
    chosen = torch.zeros_like(logits).scatter(1, logits.topk(top, 1).indices, 1.0)
    weights = chosen * (logits.exp() if score == "chosen" else torch.sigmoid(logits))
    weights = weights / weights.sum(1, keepdim=True)
    want = 0.0
    for e in range(experts):
        units = rounded(act(x @ held[f"up_{e}"].double().t()))
        want = want + rounded(weights[:, e:e + 1] * units) @ held[f"down_{e}"].double().t()
    if shared_ff:
        want = want + rounded(act(x @ held["shared_up"].double().t())) @ held["shared_down"].double().t()
    # 32-bit arithmetic in front of a rounding takes one value in some ten thousand to the other side of it: room for one in a
    # hundred, each a step of 2^-8; units that are not rounded again are off by a third of such a step each, 1e-3 in all
    assert float((got - want).norm() / want.norm()) < (1 / 100) ** 0.5 * 2.0 ** -8
