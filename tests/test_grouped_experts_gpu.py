"""Experts run on the rows that use them, against every expert on every row in 64 bits."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K
from burn_transformers_amd.parts import lookup
from burn_transformers_amd.parts.base import ResidualStream

from step_helpers import make_step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def unit_of(kind, g, u, limit):
    if kind == "gated" and limit is not None:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(1.5 * g) * (u + 1.0)
    if kind == "gated":
        return g * torch.sigmoid(g) * u
    return {"gelu_erf": torch.nn.functional.gelu(u), "silu": u * torch.sigmoid(u), "squared_relu": u.clamp(min=0.0) ** 2}[kind]


# rows around a tile's 64 and 128, experts that nobody chose and one that all chose (its list is all rows), identity
# experts among a row's choices (`zero`: weights that are exactly zero although chosen), a shared expert of another
# width with and without its gate, widths of one tile and of several that are not whole
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("tokens,width,experts,top,ff,shared_ff,identity,kind,limit,mix,skew", [
    (65, 64, 8, 2, 64, 0, 0, "gated", None, False, "even"), (129, 128, 4, 2, 192, 128, 1, "gated", None, True, "even"),
    (300, 192, 8, 1, 64, 64, 0, "squared_relu", None, False, "one"), (520, 64, 8, 3, 128, 192, 2, "gelu_erf", None, True, "even"),
    (1000, 64, 16, 4, 64, 0, 0, "gated", 2.0, False, "one"), (257, 320, 5, 2, 320, 64, 0, "silu", None, False, "zero"),
    (700, 64, 4, 2, 64, 0, 0, "gated", None, False, "one")])
def test_experts_on_their_rows(dtype, tokens, width, experts, top, ff, shared_ff, identity, kind, limit, mix, skew):
    gen = torch.Generator().manual_seed(tokens + width + experts)
    dt, outputs = DTYPES[dtype], experts + identity
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(dt).double()
    scale = width ** -0.5
    tensors = {"router": torch.zeros(outputs, width)}
    made = {}
    for e in list(range(experts)) + (["shared"] if shared_ff else []):
        inner = shared_ff if e == "shared" else ff
        name = (lambda role: f"shared_{role}") if e == "shared" else (lambda role: f"{role}_{e}")
        made[e] = [(draw(inner, width) * scale).to(dt).double(), (draw(inner, width) * scale).to(dt).double(), (draw(width, inner) * inner ** -0.5).to(dt).double()]
        for role, tensor in zip(("gate", "up", "down"), made[e]):
            if role != "gate" or kind == "gated":
                tensors[name(role)] = tensor.to(dt)
    if mix:
        tensors["shared_mix"] = torch.zeros(1, width)
    params = {"width": width, "experts": experts, "ff": ff, "identity": identity, "top": top, "shared_ff": shared_ff, "limit": limit,
              "alpha": 1.5, "unit": kind}
    part = lookup("feed_forward", "routed_experts")(params, {k: v.to(DEV) for k, v in tensors.items()})
    h = draw(tokens, width)
    # weights as the router leaves them: `top` of a row's outputs, the others zero
    scores = torch.rand(tokens, outputs, generator=gen)
    if skew == "one":                                                   # everybody chooses expert 1, nobody expert 2
        scores[:, 1], scores[:, 2] = 2.0, -1.0
    chosen = scores.topk(top, -1).indices
    weights = torch.zeros(tokens, outputs).scatter_(1, chosen, torch.rand(tokens, top, generator=gen) + 0.1)
    if skew == "zero":
        weights[::7] = 0.0
    gate = torch.rand(tokens, 1, generator=gen) if mix else None
    want = torch.zeros(tokens, width, dtype=torch.float64)
    for e in range(experts):
        g, u, d = made[e]
        want += weights[:, e:e + 1].double() * (unit_of(kind, h @ g.T, h @ u.T, limit) @ d.T)
    want += weights[:, experts:].double().sum(1, keepdim=True) * h
    if shared_ff:
        g, u, d = made["shared"]
        out = unit_of(kind, h @ g.T, h @ u.T, limit) @ d.T
        want += out * (gate.double() if mix else 1.0)
    step = make_step(dt, [tokens])
    planes = torch.full((top + (1 if shared_ff else 0), tokens + 3, width), float("nan"), device=DEV)[:, :tokens]
    assert K.groups_experts(tokens, experts, top, ff, shared_ff, width, dt) == (2 * top <= experts)
    used = ((weights != 0).long() << torch.arange(outputs)).sum(1).to(DEV)
    K.grouped_experts(h.to(dt).to(DEV), weights.to(DEV), used, None if gate is None else gate.to(DEV), part.in_weight, part.down_weight,
                      experts, ff, shared_ff, identity, top, step, planes, limit=limit, alpha=1.5, unit=None if kind == "gated" else kind)
    got = planes.sum(0).cpu().double()
    error = float((got - want).abs().max() / want.abs().max())
    # units rounded once to the products' type; sums of a few hundred 32-bit products
    assert error < (3e-6 if dtype == "float32" else 8e-3), error


def test_a_part_takes_them_in_steps_of_many_tokens(monkeypatch):
    """The part's two ways give the same sums, in steps on both sides of the rule."""
    monkeypatch.setattr(K, "GROUPED_SAVED", 0.0)              # (however little there is to save)
    monkeypatch.setattr(K, "GROUPED_SAVED_A_PLANE", 0.0)
    gen = torch.Generator().manual_seed(3)
    width, experts, ff = 128, 8, 128
    tensors = {"router": torch.randn(experts, width, generator=gen) * 0.1}
    for e in range(experts):
        for role, shape in (("gate", (ff, width)), ("up", (ff, width)), ("down", (width, ff))):
            tensors[f"{role}_{e}"] = (torch.randn(shape, generator=gen) * 0.1).to(torch.bfloat16)
    part = lookup("feed_forward", "routed_experts")({"width": width, "experts": experts, "ff": ff, "top": 2}, {k: v.to(DEV) for k, v in tensors.items()})
    for tokens in (64, 65, 200):
        h = torch.randn(tokens, width, generator=gen).to(torch.bfloat16).to(DEV)
        sums = []
        for way in (True, False):
            K.GROUPED_EXPERTS = way
            try:
                delta = part.forward(h, make_step(torch.bfloat16, [tokens]), ResidualStream(torch.zeros(tokens, width, device=DEV)))
                sums.append(delta.partials.sum(0).cpu().double())
            finally:
                K.GROUPED_EXPERTS = True
        assert float((sums[0] - sums[1]).abs().max() / sums[1].abs().max()) < 1.2e-2


# steps on both sides of 1,536 tokens, from which on sixteen tokens share a work-group where the outputs fill at most two tiles of
# sixteen: tokens that are no multiple of sixteen, outputs of one tile, of just two (by an expert or by the gate beside sixteen) and of
# both whole, a gate beside them, groups, every kind of score, corrections and biases, rows that lie apart.  The choice itself is
# that of the kernel with a work-group a token, which every step of 100 tokens takes
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("tokens,width,outputs,top,groups,keep,score,rank,normalize,extras", [
    (128, 64, 8, 2, 1, 1, "softmax", 1, True, ""), (333, 1024, 9, 2, 3, 2, "softmax", 1, True, "correction gate"),
    (150, 48, 16, 4, 4, 2, "sigmoid", 2, False, "gate"), (200, 80, 33, 3, 1, 1, "chosen", 1, True, "bias"), (129, 16, 64, 8, 8, 3, "softmax", 1, True, "correction bias"),
    (1536, 16, 1, 1, 1, 1, "softmax", 1, False, "gate"), (1537, 64, 8, 2, 1, 1, "softmax", 1, True, ""),
    (1809, 1024, 9, 2, 3, 2, "softmax", 1, True, "correction gate"), (2447, 48, 16, 4, 4, 2, "sigmoid", 2, False, "gate"),
    (1551, 96, 16, 2, 1, 1, "softmax", 1, True, "bias"), (1552, 80, 17, 3, 1, 1, "chosen", 1, True, "bias"),
    (1600, 1040, 32, 8, 8, 3, "softmax", 1, True, "correction bias"), (1539, 2048, 31, 4, 1, 1, "sigmoid", 1, True, "correction gate")])
def test_router_of_many_tokens(dtype, tokens, width, outputs, top, groups, keep, score, rank, normalize, extras):
    gen = torch.Generator().manual_seed(tokens + outputs)
    h = torch.randn(tokens, width + 8, generator=gen).to(DTYPES[dtype]).to(DEV)[:, :width]
    router = (torch.randn(outputs, width, generator=gen) * width ** -0.5).to(DEV)
    correction = (torch.randn(outputs, generator=gen) * 0.1).to(DEV) if "correction" in extras else None
    bias = torch.randn(outputs, generator=gen).to(DEV) if "bias" in extras else None
    mix = torch.randn(width, generator=gen).to(DEV) if "gate" in extras else None
    many, few = [dict(weights=torch.full((tokens, outputs), float("nan"), device=DEV), gate=torch.full((tokens, 1), float("nan"), device=DEV),
                      used=torch.zeros(tokens, dtype=torch.int64, device=DEV)) for _ in range(2)]
    run = lambda rows, to, part: K.route(rows, router, correction, top, groups, keep, to["weights"][part], mix, to["gate"][part] if mix is not None else None,
                                         score=score, group_rank=rank, normalize=normalize, bias=bias, used=to["used"][part])
    run(h, many, slice(0, tokens))
    for begin in range(0, tokens, 100):
        part = slice(begin, min(begin + 100, tokens))
        run(h[part], few, part)
    assert torch.equal((many["weights"] != 0), (few["weights"] != 0))
    # logits of size one from sums of `width` products in another order
    assert float((many["weights"] - few["weights"]).abs().max()) < 4e-6
    # the chosen experts' weights in 64 bits
    logits = h.double().cpu() @ router.double().cpu().T + (bias.double().cpu() if bias is not None else 0.0)
    mask = (few["weights"] != 0).cpu()
    if score == "chosen":
        exact = logits.masked_fill(~mask, float("-inf")).softmax(-1)
    else:
        exact = torch.where(mask, logits.softmax(-1) if score == "softmax" else logits.sigmoid(), 0.0)
        exact = exact / exact.sum(1, keepdim=True) if normalize else exact
    assert float((many["weights"].cpu().double() - exact).abs().max()) < 4e-6
    want = ((many["weights"] != 0).long() << torch.arange(outputs, device=DEV)).sum(1)
    assert torch.equal(many["used"], want) and torch.equal(few["used"], want)
    if mix is not None:
        # (the gate's row is of size one: where the gate is steep the parts of its sum are about sqrt(width) large and take some fifty
        # roundings, sqrt(50) of 2^-24, of which the sigmoid passes a quarter; four times that)
        bound = 4e-6 if width <= 1024 else 7 * 2.0 ** -24 * width ** 0.5
        assert float((many["gate"] - few["gate"]).abs().max()) < bound
        exact = torch.sigmoid(h.double() @ mix.double())
        assert float((many["gate"][:, 0].double() - exact).abs().max()) < bound


def chosen_by(scores, corrected, top, groups, keep):
    """[rows, outputs] of booleans: the ``top`` largest corrected scores (the lower index among equals) in the ``keep`` groups
    with the largest best."""
    rows, outputs = scores.shape
    if groups > 1:
        best = corrected.view(rows, groups, -1).amax(-1)
        kept = best.sort(dim=-1, descending=True, stable=True).indices[:, :keep]
        open_ = torch.zeros(rows, groups, dtype=torch.bool).scatter_(1, kept, True).repeat_interleave(outputs // groups, 1)
        corrected = corrected.masked_fill(~open_, float("-inf"))
    order = corrected.sort(dim=-1, descending=True, stable=True).indices[:, :top]
    return torch.zeros(rows, outputs, dtype=torch.bool).scatter_(1, order, True)


# a correction or a logit without end is one choice like any other and no sign of one that was made: never more than `top`
# experts, however many there are of them, in every kernel that makes the choice
@pytest.mark.parametrize("tokens", [3, 64, 200, 1537])
@pytest.mark.parametrize("score,groups,keep,endless", [
    ("softmax", 1, 1, [5]), ("softmax", 1, 1, [0, 2, 3, 7]), ("sigmoid", 4, 2, [5]), ("softmax", 4, 2, [1, 6]), ("chosen", 1, 1, [2, 4, 6])])
def test_endless_corrections_are_choices_like_others(tokens, score, groups, keep, endless):
    gen = torch.Generator().manual_seed(tokens + len(endless))
    width, outputs, top = 64, 8, 2
    h = torch.randn(tokens, width, generator=gen)
    router = torch.randn(outputs, width, generator=gen) * width ** -0.5
    extra = torch.randn(outputs, generator=gen) * 0.1
    extra[endless] = float("inf")
    logits = h.double() @ router.double().T
    scores = {"softmax": logits.softmax(-1), "sigmoid": logits.sigmoid(), "chosen": logits}[score]
    mask = chosen_by(scores, scores + extra.double(), top, groups, keep)
    assert bool((mask.sum(1) == top).all())
    weights, used = torch.full((tokens, outputs), -1.0, device=DEV), torch.zeros(tokens, dtype=torch.int64, device=DEV)
    # (a "chosen" score weighs by the logits with their bias: of infinite ones nobody knows the softmax)
    more = {"bias": extra.to(DEV)} if score == "chosen" else {}
    K.route(h.to(DEV), router.to(DEV), None if more else extra.to(DEV), top, groups, keep, weights, score=score, used=used, **more)
    got = weights.cpu()
    assert torch.equal(got != 0, mask)                                  # (not a number is not zero)
    assert torch.equal(used.cpu(), (mask.long() << torch.arange(outputs)).sum(1))
    if score != "chosen":
        want = torch.where(mask, scores, 0.0)
        assert float((got.double() - want / want.sum(1, keepdim=True)).abs().max()) < 4e-6


def test_a_part_with_an_endless_correction_on_both_sides_of_the_rule():
    gen = torch.Generator().manual_seed(5)
    width, experts, ff = 128, 8, 128
    correction = torch.randn(experts, generator=gen) * 0.1
    correction[3] = float("inf")
    tensors = {"router": torch.randn(experts, width, generator=gen) * 0.1, "correction": correction}
    for e in range(experts):
        for role, shape in (("gate", (ff, width)), ("up", (ff, width)), ("down", (width, ff))):
            tensors[f"{role}_{e}"] = torch.randn(shape, generator=gen) * 0.1
    part = lookup("feed_forward", "routed_experts")({"width": width, "experts": experts, "ff": ff, "top": 2}, {k: v.to(DEV) for k, v in tensors.items()})
    h = torch.randn(200, width, generator=gen)
    scores = (h.double() @ tensors["router"].double().T).softmax(-1)
    weights = torch.where(chosen_by(scores, scores + correction.double(), 2, 1, 1), scores, 0.0)
    weights /= weights.sum(1, keepdim=True)
    want = sum(weights[:, e:e + 1] * (unit_of("gated", h.double() @ tensors[f"gate_{e}"].double().T, h.double() @ tensors[f"up_{e}"].double().T, None)
                                      @ tensors[f"down_{e}"].double().T) for e in range(experts))
    for tokens in (1, 64, 65, 200):
        delta = part.forward(h[:tokens].to(DEV), make_step(torch.float32, [tokens]), ResidualStream(torch.zeros(tokens, width, device=DEV)))
        got = delta.partials.sum(0).cpu().double()
        # sums of 128 products of 32-bit values, two of them one behind the other
        assert float((got - want[:tokens]).abs().max() / want.abs().max()) < 5e-6


def test_a_token_has_room_for_its_choices_only():
    """Words that name more than ``top`` experts: the first ``top`` of them count, and no plane behind theirs is touched."""
    gen = torch.Generator().manual_seed(6)
    tokens, width, experts, ff, top = 130, 64, 8, 64, 2
    matrices = [[torch.randn(ff, width, generator=gen) * 0.1, torch.randn(ff, width, generator=gen) * 0.1, torch.randn(width, ff, generator=gen) * 0.1] for _ in range(experts)]
    tensors = {"router": torch.zeros(experts, width)}
    for e, made in enumerate(matrices):
        tensors.update({f"{role}_{e}": m for role, m in zip(("gate", "up", "down"), made)})
    part = lookup("feed_forward", "routed_experts")({"width": width, "experts": experts, "ff": ff, "top": top}, {k: v.to(DEV) for k, v in tensors.items()})
    h = torch.randn(tokens, width, generator=gen)
    named = torch.rand(tokens, experts, generator=gen).topk(4, -1).indices
    weights = torch.zeros(tokens, experts).scatter_(1, named, torch.rand(tokens, 4, generator=gen) + 0.1)
    used = ((weights != 0).long() << torch.arange(experts)).sum(1)
    first = (weights != 0) & ((weights != 0).cumsum(1) <= top)
    planes = torch.full((top + 1, tokens, width), float("nan"), device=DEV)
    step = make_step(torch.float32, [tokens])
    K.grouped_experts(h.to(DEV), weights.to(DEV), used.to(DEV), None, part.in_weight, part.down_weight, experts, ff, 0, 0, top, step, planes[:top])
    want = sum(torch.where(first, weights, 0.0)[:, e:e + 1].double() * (unit_of("gated", h.double() @ g.double().T, h.double() @ u.double().T, None) @ d.double().T)
               for e, (g, u, d) in enumerate(matrices))
    assert float((planes[:top].sum(0).cpu().double() - want).abs().max() / want.abs().max()) < 5e-6
    assert bool(torch.isnan(planes[top]).all())
