"""The selective scan with a channel a lane, the keyed scan and the scan with one decay a head in blocks of sixteen tokens on the matrix units, against the recurrence token by token in 64 bits."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

from step_helpers import make_step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rel_err(got, want):
    return float((got.double() - want).abs().max() / want.abs().max())


def recurrence(S, q, k, v, decay, beta):
    """S [H, D, V]; rows [T, H, ...] in 64 bits: (read-outs [T, H, V], the state behind them)."""
    out = []
    for t in range(q.shape[0]):
        S = decay[t][..., None] * S
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - (S * k[t][..., None]).sum(1))
        S = S + k[t][..., None] * u[:, None]
        out.append((S * q[t][..., None]).sum(1))
    return torch.stack(out), S


def state_rows(state, heads, dim, vdim):
    """A slot's floats as [heads, dim, vdim]."""
    return state[:, :heads * dim * vdim].view(-1, heads, vdim // 4, dim, 4).permute(0, 1, 3, 2, 4).reshape(-1, heads, dim, vdim)


# lengths around a block's edges beside the shortest and sequences of one token; a second portion starts from a state
# that is not zero; `strong`: decays down to nothing (products that underflow) beside decays of nearly one
@pytest.mark.parametrize("form,heads,kv_heads,dim,vdim,lengths,strong", [
    ("head", 4, 2, 128, 128, [33, 1, 16, 47], False), ("head", 2, 2, 16, 16, [100, 32, 5], True),
    ("channel", 2, 1, 128, 32, [64, 17, 31], False), ("channel", 3, 3, 80, 48, [49, 2], True),
    ("forget", 2, 2, 128, 128, [130, 15, 1], False), ("forget", 3, 3, 48, 80, [35, 64], True),
    ("channel", 1, 1, 64, 16, [400], False), ("forget", 1, 1, 32, 64, [333], True), ("head", 2, 2, 32, 32, [300] + [1] * 70 + [20], False),
    ("forget", 2, 2, 32, 16, [1] * 64 + [300, 16, 1], False)])
def test_blocks_of_tokens(form, heads, kv_heads, dim, vdim, lengths, strong):
    gen = torch.Generator().manual_seed(heads * 1000 + dim + len(lengths))
    qk, inner = kv_heads * dim, heads * vdim
    decays = heads if form == "head" else heads * dim
    columns = 2 * qk + inner + decays + heads + 3                       # an odd pitch: rows are not aligned
    portions = [lengths, [n % 40 + 32 for n in lengths]]
    A_log, bias = torch.log(torch.rand(heads, generator=gen) * 3.0 + 0.5), torch.randn(decays, generator=gen)
    lower = torch.rand(decays, generator=gen) * (0.0 if strong else 0.9)
    slots = list(reversed(range(len(lengths))))
    state = torch.zeros(len(lengths), heads * dim * vdim + 7, device=DEV)
    walked = state.clone()
    want_state = [torch.zeros(heads, dim, vdim, dtype=torch.float64) for _ in lengths]
    spread = lambda x: x.repeat_interleave(heads // kv_heads, 1)
    errors = {"blocks": [], "walk": []}
    for part, counts in enumerate(portions):
        rows = torch.randn(sum(counts), columns, generator=gen)
        if strong:
            rows[:, 2 * qk + inner:2 * qk + inner + decays] *= 20.0
        r = rows.double()
        q, k = r[:, :qk].view(-1, kv_heads, dim), r[:, qk:2 * qk].view(-1, kv_heads, dim)
        v, raw = r[:, 2 * qk:2 * qk + inner].view(-1, heads, vdim), r[:, 2 * qk + inner:2 * qk + inner + decays]
        beta = None
        if form == "forget":
            decay = (lower.double() + (1.0 - lower.double()) * torch.sigmoid(raw + bias.double())).view(-1, heads, dim)
            q, k = (q * torch.sigmoid(q)), 1.0 - decay
        else:
            unit = lambda x: spread(x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6))
            q, k, beta = unit(q) * dim ** -0.5, unit(k), torch.sigmoid(r[:, -3 - heads:-3])
            dt = torch.nn.functional.softplus(raw + bias.double(), threshold=50.0).view(-1, heads, decays // heads)
            decay = torch.exp(-torch.exp(A_log.double())[:, None] * dt).expand(-1, heads, dim)
        step = make_step(torch.float32, counts, starts=[0 if part == 0 else n for n in lengths], slots=slots)
        on = rows.to(DEV)
        run = dict(blocks=(state, K.scan_blocks(step, heads, dim, vdim)), walk=(walked, None))
        assert run["blocks"][1] is not None
        want, at = [], 0
        for s, n in enumerate(counts):
            here = slice(at, at + n)
            o, want_state[s] = recurrence(want_state[s], q[here], k[here], v[here], decay[here], None if beta is None else beta[here])
            want.append(o.reshape(n, inner))
            at += n
        want = torch.cat(want)
        for name, (held, room) in run.items():
            y = torch.full((sum(counts), inner + 2), float("nan"), device=DEV)
            if room is not None:
                room.fill_(float("nan"))
            extra = dict(g_bias=bias.to(DEV), lower=lower.to(DEV)) if form == "forget" else \
                dict(beta=on[:, -3 - heads:-3], A_log=A_log.to(DEV), unit=True, unit_eps=1e-6, q_scale=dim ** -0.5,
                     decay_per_head=form == "head", dt_bias=bias.to(DEV))
            K.keyed_scan(on[:, :qk], None if form == "forget" else on[:, qk:2 * qk], on[:, 2 * qk:2 * qk + inner],
                         on[:, 2 * qk + inner:2 * qk + inner + decays], y, held, step, heads, kv_heads, dim, vdim,
                         "forget" if form == "forget" else "delta", blocks=room, **extra)
            assert bool(torch.isnan(y[:, inner:]).all())
            errors[name].append(rel_err(y[:, :inner].cpu(), want))
            got = state_rows(held, heads, dim, vdim).cpu()
            errors[name].append(max(rel_err(got[slot], w) for slot, w in zip(slots, want_state)))
    # a sum of 128 products of 32-bit values and a few hundred decays multiplied one after the other: some 1e-6
    assert max(errors["blocks"]) < 5e-6, errors
    assert max(errors["blocks"]) < 3.0 * max(errors["walk"]), errors


# the forget gate with room for spans: spans of 64 tokens and of more, two and many of a sequence, a last one of one token and whole,
# sequences too short to be cut beside them, key channels that are no multiple of the waves' tiles
@pytest.mark.parametrize("heads,dim,vdim,lengths,strong", [
    (2, 128, 128, [705, 15, 1, 640], False), (3, 48, 80, [640, 127, 193], True), (1, 64, 16, [700, 64], False), (4, 80, 32, [1, 833, 1, 1], True),
    (8, 128, 128, [1100, 90, 1030], False)])
def test_blocks_of_tokens_in_spans(heads, dim, vdim, lengths, strong):
    gen = torch.Generator().manual_seed(heads * 1000 + dim + len(lengths))
    qk, inner, total = heads * dim, heads * vdim, sum(lengths)
    rows = torch.randn(total, 2 * qk + inner + 3, generator=gen)
    rows[:, qk:2 * qk] *= 20.0 if strong else 1.0
    bias, lower = torch.randn(qk, generator=gen), torch.rand(qk, generator=gen) * (0.0 if strong else 0.9)
    slots = list(reversed(range(len(lengths))))
    state = torch.randn(len(lengths), qk * vdim, generator=gen)
    step, on, held = make_step(torch.float32, lengths, starts=[5] * len(lengths), slots=slots), rows.to(DEV), state.to(DEV)
    blocks, carry = K.scan_blocks(step, heads, dim, vdim), K.scan_carry(step, qk * vdim, qk)
    blocks.fill_(float("nan"))
    carry.fill_(float("nan"))
    y = torch.full((total, inner + 2), float("nan"), device=DEV)
    K.keyed_scan(on[:, :qk], None, on[:, 2 * qk:2 * qk + inner], on[:, qk:2 * qk], y, held, step, heads, heads, dim, vdim, "forget",
                 g_bias=bias.to(DEV), lower=lower.to(DEV), carry=carry, blocks=blocks)
    assert bool(torch.isnan(y[:, inner:]).all())
    assert bool(torch.isfinite(carry).any()) and bool(torch.isfinite(blocks).any())             # (cut indeed, and in blocks)
    r, q = rows.double(), rows[:, :qk].double()
    decay = (lower.double() + (1.0 - lower.double()) * torch.sigmoid(r[:, qk:2 * qk] + bias.double())).view(-1, heads, dim)
    q, v, at, want, got = (q * torch.sigmoid(q)).view(-1, heads, dim), r[:, 2 * qk:2 * qk + inner].view(-1, heads, vdim), 0, [], state_rows(held, heads, dim, vdim).cpu()
    for slot, n in zip(slots, lengths):
        here = slice(at, at + n)
        o, behind = recurrence(state_rows(state, heads, dim, vdim)[slot].double(), q[here], 1.0 - decay[here], v[here], decay[here], None)
        want.append(o.reshape(n, inner))
        assert rel_err(got[slot], behind) < 5e-6                # (as in whole sequences: the spans' products are a few more of some hundred)
        at += n
    assert rel_err(y[:, :inner].cpu(), torch.cat(want)) < 5e-6


# which steps are cut: one sequence from 640 tokens on, several that fill half the compute units from 832 on
@pytest.mark.parametrize("heads,dim,vdim,lengths,cut", [
    (8, 128, 128, [640], True), (8, 128, 128, [639], False), (8, 128, 128, [640, 640], False), (8, 128, 128, [831, 640], False), (8, 128, 128, [832, 640], True),
    (4, 128, 128, [640] * 4, False), (4, 128, 128, [640, 640], True), (16, 128, 128, [640], True)])
def test_which_steps_are_cut_into_spans(heads, dim, vdim, lengths, cut):
    qk, total = heads * dim, sum(lengths)
    step = make_step(torch.float32, lengths)
    rows, y = torch.randn(total, 2 * qk + heads * vdim, device=DEV), torch.empty(total, heads * vdim, device=DEV)
    blocks, carry = K.scan_blocks(step, heads, dim, vdim), K.scan_carry(step, qk * vdim, qk)
    blocks.fill_(float("nan"))
    carry.fill_(float("nan"))
    K.keyed_scan(rows[:, :qk], None, rows[:, 2 * qk:], rows[:, qk:2 * qk], y, torch.zeros(len(lengths), qk * vdim, device=DEV), step, heads, heads, dim, vdim,
                 "forget", g_bias=torch.zeros(qk, device=DEV), lower=torch.rand(qk, device=DEV), carry=carry, blocks=blocks)
    assert bool(torch.isfinite(blocks).any())                                                   # (in blocks, not token by token)
    assert bool(torch.isfinite(carry).any()) == cut


# one token of one sequence whose operand is not finite, in the middle of a block and at its end: earlier tokens and other
# sequences do not see it, later ones as in the walk (an endless step is a decay of nothing and stays finite)
@pytest.mark.parametrize("form,where,value", [
    (form, where, value) for form in ("head", "channel", "forget")
    for where, value in (("v", "inf"), ("v", "nan"), ("k", "inf"), ("k", "nan"), ("q", "inf"), ("g", "nan"), ("g", "inf"), ("beta", "nan"))
    if form != "forget" or where not in ("k", "beta")])                 # (the forget gate has no such operands)
@pytest.mark.parametrize("token", [21, 31, 39])
def test_a_token_that_is_not_finite_spoils_no_earlier_one(form, where, value, token):
    gen = torch.Generator().manual_seed(7)
    heads, dim, vdim, lengths = 2, 64, 32, [40, 50]
    qk, inner = heads * dim, heads * vdim
    decays = heads if form == "head" else heads * dim
    total = sum(lengths)
    A_log, bias, lower = torch.zeros(heads, device=DEV), torch.randn(decays, generator=gen).to(DEV), (torch.rand(decays, generator=gen) * 0.9).to(DEV)
    rows = torch.randn(total, 2 * qk + inner + decays + heads, generator=gen)
    at = {"q": 3, "k": qk + 3, "v": 2 * qk + 3, "g": 2 * qk + inner, "beta": 2 * qk + inner + decays}[where]
    spoiled = rows.clone()
    spoiled[token, at] = float(value)
    step = make_step(torch.float32, lengths)
    results = {}
    for name, source, blocked in (("clean", rows, True), ("blocks", spoiled, True), ("walk", spoiled, False)):
        on, state = source.to(DEV), torch.zeros(len(lengths), heads * dim * vdim, device=DEV)
        y = torch.full((total, inner), -7.0, device=DEV)
        extra = dict(g_bias=bias, lower=lower) if form == "forget" else \
            dict(beta=on[:, -heads:], A_log=A_log, unit=False, q_scale=1.0, decay_per_head=form == "head", dt_bias=bias)
        if form != "forget":
            on[:, :2 * qk] *= dim ** -0.5
        K.keyed_scan(on[:, :qk], None if form == "forget" else on[:, qk:2 * qk], on[:, 2 * qk:2 * qk + inner], on[:, 2 * qk + inner:2 * qk + inner + decays],
                     y, state, step, heads, heads, dim, vdim, "forget" if form == "forget" else "delta",
                     blocks=K.scan_blocks(step, heads, dim, vdim) if blocked else None, **extra)
        results[name] = (y.cpu(), state.cpu())
    (clean, _), (blocks, state), (walk, walked) = results["clean"], results["blocks"], results["walk"]
    # (a block with such a token sums in another order: a few roundings of 32 bits)
    assert rel_err(blocks[:token], clean[:token].double()) < 2e-6
    assert torch.equal(blocks[lengths[0]:], clean[lengths[0]:])
    assert torch.equal(torch.isfinite(blocks), torch.isfinite(walk)) and torch.equal(torch.isfinite(state), torch.isfinite(walked))
    assert bool(torch.isfinite(blocks).all()) == (where == "g" and value == "inf")
    kept = torch.isfinite(walk)
    assert rel_err(blocks[kept], walk[kept].double()) < 1e-5


# the same where the sequence is cut into spans: a token of the first span, of one between, at a span's end and of the last; the walk token by token is whole
@pytest.mark.parametrize("where,value", [("v", "inf"), ("v", "-inf"), ("v", "nan"), ("q", "inf"), ("q", "nan"), ("g", "nan"), ("g", "inf"), ("g", "-inf")])
@pytest.mark.parametrize("token", [5, 250, 255, 699])
def test_a_token_that_is_not_finite_in_a_cut_sequence(where, value, token):
    gen = torch.Generator().manual_seed(9)
    heads, dim, vdim, lengths = 4, 128, 64, [700, 650]
    qk, inner, total = heads * dim, heads * vdim, sum(lengths)
    bias, lower = torch.randn(qk, generator=gen).to(DEV), (torch.rand(qk, generator=gen) * 0.9).to(DEV)
    rows = torch.randn(total, 2 * qk + inner, generator=gen)
    spoiled = rows.clone()
    spoiled[token, {"q": 3, "g": qk + 3, "v": 2 * qk + 3}[where]] = float(value)
    step, results = make_step(torch.float32, lengths), {}
    for name, source, blocked in (("clean", rows, True), ("spans", spoiled, True), ("walk", spoiled, False)):
        on, state = source.to(DEV), torch.zeros(len(lengths), qk * vdim, device=DEV)
        y = torch.full((total, inner), -7.0, device=DEV)
        blocks, carry = (K.scan_blocks(step, heads, dim, vdim).fill_(float("nan")), K.scan_carry(step, qk * vdim, qk).fill_(float("nan"))) if blocked else (None, None)
        K.keyed_scan(on[:, :qk], None, on[:, 2 * qk:], on[:, qk:2 * qk], y, state, step, heads, heads, dim, vdim, "forget", g_bias=bias, lower=lower, carry=carry,
                     blocks=blocks)
        assert not blocked or (bool(torch.isfinite(blocks).any()) and bool(torch.isfinite(carry).any()))
        results[name] = (y.cpu(), state.cpu())
    (clean, _), (spans, state), (walk, walked) = results["clean"], results["spans"], results["walk"]
    # (a block with such a token sums in another order: a few roundings of 32 bits)
    assert rel_err(spans[:token], clean[:token].double()) < 2e-6
    assert torch.equal(spans[lengths[0]:], clean[lengths[0]:])
    assert torch.equal(torch.isfinite(spans), torch.isfinite(walk)) and torch.equal(torch.isfinite(state), torch.isfinite(walked))
    assert bool(torch.isfinite(spans).all()) == (where == "g" and value != "nan")
    kept = torch.isfinite(walk)
    assert rel_err(spans[kept], walk[kept].double()) < 1e-5


@pytest.mark.parametrize("heads,groups,vdim,state,lengths,strong", [
    (4, 1, 64, 128, [33, 1, 16, 47], False), (12, 1, 16, 16, [100, 32, 5], True), (6, 3, 48, 80, [49, 2], False),
    (9, 1, 32, 48, [400], True), (2, 2, 16, 32, [64, 63, 65], False), (20, 2, 16, 128, [333, 17], False), (4, 1, 32, 32, [300] + [1] * 70 + [20], False)])
def test_heads_in_blocks_of_tokens(heads, groups, vdim, state, lengths, strong):
    gen = torch.Generator().manual_seed(heads * 1000 + state + len(lengths))
    inner, bc = heads * vdim, groups * state
    columns = inner + 2 * bc + heads + 1                                # an odd pitch
    A_log, bias, D = torch.log(torch.rand(heads, generator=gen) * 7.0 + 1.0), torch.randn(heads, generator=gen) - 2.0, torch.randn(heads, generator=gen)
    slots = list(reversed(range(len(lengths))))
    held = torch.zeros(len(lengths), heads * state * vdim + 7, device=DEV)
    walked = held.clone()
    want_state = [torch.zeros(heads, state, vdim, dtype=torch.float64) for _ in lengths]
    errors = {"blocks": [], "walk": []}
    for part, counts in enumerate([lengths, [n % 40 + 40 for n in lengths]]):
        rows = torch.randn(sum(counts), columns, generator=gen)
        if strong:
            rows[:, inner + 2 * bc:] *= 20.0
        r, on = rows.double(), rows.to(DEV)
        spread = lambda v: v.view(-1, groups, state).repeat_interleave(heads // groups, 1)
        x, B, C = r[:, :inner].view(-1, heads, vdim), spread(r[:, inner:inner + bc]), spread(r[:, inner + bc:inner + 2 * bc])
        dt = torch.nn.functional.softplus(r[:, inner + 2 * bc:inner + 2 * bc + heads] + bias.double(), threshold=50.0)
        decay = torch.exp(-torch.exp(A_log.double()) * dt)[..., None].expand(-1, heads, state)
        step = make_step(torch.float32, counts, starts=[0 if part == 0 else n for n in lengths], slots=slots)
        want, at = [], 0
        for s, n in enumerate(counts):
            here = slice(at, at + n)
            o, want_state[s] = recurrence(want_state[s], C[here], B[here], dt[here][..., None] * x[here], decay[here], None)
            want.append((o + D.double()[:, None] * x[here]).reshape(n, inner))
            at += n
        want = torch.cat(want)
        for name, slot_rows, room in (("blocks", held, K.head_blocks(step, heads, vdim, state, groups)), ("walk", walked, None)):
            y = torch.full((sum(counts), inner + 2), float("nan"), device=DEV)
            if room is not None:
                room.fill_(float("nan"))
            K.head_scan(on[:, :inner], on[:, inner:inner + bc], on[:, inner + bc:inner + 2 * bc], on[:, inner + 2 * bc:], bias.to(DEV), A_log.to(DEV),
                        D.to(DEV), y, slot_rows, step, heads, vdim, state, groups, blocks=room)
            assert bool(torch.isnan(y[:, inner:]).all())
            errors[name].append(rel_err(y[:, :inner].cpu(), want))
            got = state_rows(slot_rows, heads, state, vdim).cpu()
            errors[name].append(max(rel_err(got[slot], w) for slot, w in zip(slots, want_state)))
    assert max(errors["blocks"]) < 5e-6, errors
    assert max(errors["blocks"]) < 3.0 * max(errors["walk"]), errors


# read-outs of heads in blocks against 64 bits, in the 2-norm: as exact as token by token (their roundings differ by some hundredths; one
# chain of 32 products a wave for the blocks' C B^T was a third further off)
@pytest.mark.parametrize("state", [64, 128])
@pytest.mark.parametrize("shift", [-2.0, 0.5])
def test_heads_in_blocks_are_as_exact(state, shift):
    gen, heads, vdim, total = torch.Generator().manual_seed(11), 8, 64, 500
    inner = heads * vdim
    rows = torch.randn(total, inner + 2 * state + heads, generator=gen)
    A_log, bias, D = torch.log(torch.rand(heads, generator=gen) * 15.0 + 1.0), torch.randn(heads, generator=gen) * 0.5 + shift, torch.ones(heads)
    r, on, step = rows.double(), rows.to(DEV), make_step(torch.float32, [total])
    x, B, C = r[:, :inner].view(-1, heads, vdim), r[:, None, inner:inner + state], r[:, None, inner + state:inner + 2 * state]
    dt = torch.nn.functional.softplus(r[:, inner + 2 * state:] + bias.double(), threshold=50.0)
    decay = torch.exp(-torch.exp(A_log.double()) * dt)[..., None].expand(-1, heads, state)
    want, _ = recurrence(torch.zeros(heads, state, vdim, dtype=torch.float64), C.expand(-1, heads, -1), B.expand(-1, heads, -1), dt[..., None] * x, decay, None)
    want = (want + x).reshape(total, inner)
    errors = []
    for room in (K.head_blocks(step, heads, vdim, state, 1), None):
        y, held = torch.empty(total, inner, device=DEV), torch.zeros(1, heads * state * vdim, device=DEV)
        K.head_scan(on[:, :inner], on[:, inner:inner + state], on[:, inner + state:inner + 2 * state], on[:, inner + 2 * state:], bias.to(DEV), A_log.to(DEV),
                    D.to(DEV), y, held, step, heads, vdim, state, 1, blocks=room)
        errors.append(float((y.double().cpu() - want).norm() / want.norm()))
    assert errors[0] < 1.15 * errors[1], errors


# the same for the scan with one decay a head
@pytest.mark.parametrize("where,value", [("x", "inf"), ("x", "-inf"), ("x", "nan"), ("B", "inf"), ("B", "nan"), ("C", "inf"), ("dt", "nan"), ("dt", "inf")])
@pytest.mark.parametrize("token", [0, 21, 31, 38, 39])
def test_a_token_that_is_not_finite_spoils_no_earlier_one_of_a_head(where, value, token):
    gen = torch.Generator().manual_seed(8)
    heads, vdim, state, lengths = 2, 32, 64, [40, 50]
    inner, total = heads * vdim, sum(lengths)
    A_log, bias, D = torch.zeros(heads, device=DEV), torch.randn(heads, generator=gen).to(DEV), torch.randn(heads, generator=gen).to(DEV)
    rows = torch.randn(total, inner + 2 * state + heads, generator=gen)
    spoiled = rows.clone()
    spoiled[token, {"x": 3, "B": inner + 3, "C": inner + state + 3, "dt": inner + 2 * state}[where]] = float(value)
    step = make_step(torch.float32, lengths)
    results = {}
    for name, source, blocked in (("clean", rows, True), ("blocks", spoiled, True), ("walk", spoiled, False)):
        on, held = source.to(DEV), torch.zeros(len(lengths), heads * state * vdim, device=DEV)
        y = torch.full((total, inner), -7.0, device=DEV)
        room = K.head_blocks(step, heads, vdim, state, 1) if blocked else None
        if blocked:
            room.fill_(float("nan"))
        K.head_scan(on[:, :inner], on[:, inner:inner + state], on[:, inner + state:inner + 2 * state], on[:, inner + 2 * state:], bias, A_log, D, y, held, step,
                    heads, vdim, state, 1, blocks=room)
        assert not blocked or bool(torch.isfinite(room).any())          # (it did go in blocks)
        results[name] = (y.cpu(), held.cpu())
    (clean, _), (blocks, ended), (walk, walked) = results["clean"], results["blocks"], results["walk"]
    # (a block with such a token sums in another order: a few roundings of 32 bits)
    assert token == 0 or rel_err(blocks[:token], clean[:token].double()) < 2e-6
    assert torch.equal(blocks[lengths[0]:], clean[lengths[0]:])
    assert torch.equal(torch.isfinite(blocks), torch.isfinite(walk)) and torch.equal(torch.isfinite(ended), torch.isfinite(walked))
    assert not bool(torch.isfinite(blocks).all())
    kept = torch.isfinite(walk)
    assert rel_err(blocks[kept], walk[kept].double()) < 1e-5


# channels that do not fill a wave, all sizes of state that lanes take, steps on both sides of the rule, spans that end
# within a sequence, a second portion from a state that is not zero; `strong`: steps so long that decays vanish
@pytest.mark.parametrize("channels,state,lengths,spans,strong", [
    (100, 16, [64, 1, 130], True, False), (64, 8, [65, 63], False, True), (200, 32, [300, 17, 64], True, False), (70, 16, [500], True, True),
    (1100, 16, [20] * 16, True, False), (48, 16, [63, 5], True, False), (100, 32, [191, 64], True, False), (100, 32, [192, 2], True, True),
    (100, 24, [64, 200], True, False), (100, 16, [300] + [1] * 70 + [20], True, False), (70, 8, [1] * 64 + [200, 16, 1], True, False),
    (130, 32, [1, 400, 1, 1], True, False)])
def test_channels_in_lanes(channels, state, lengths, spans, strong):
    gen = torch.Generator().manual_seed(channels + state + len(lengths))
    A_log, D = torch.log(torch.rand(channels, state, generator=gen) * 7.0 + 0.5), torch.randn(channels, generator=gen)
    A = -torch.exp(A_log.double())
    slots = list(reversed(range(len(lengths))))
    held = torch.zeros(len(lengths), channels * state + 3, device=DEV)
    want_state = [torch.zeros(channels, state, dtype=torch.float64) for _ in lengths]
    for part, counts in enumerate([lengths, [n % 40 + 40 for n in lengths]]):
        total = sum(counts)
        rows = torch.randn(total, 3 * channels + 2 * state + 1, generator=gen)
        x, z, raw, B, C = rows.split([channels, channels, channels, state, state + 1], 1)
        dt = torch.nn.functional.softplus(raw * (20.0 if strong else 1.0) - 2.0)
        if strong:
            dt[5], x[5] = 1e30, 0.0                                     # an endless step that writes nothing leaves nothing behind
        step = make_step(torch.float32, counts, starts=[0 if part == 0 else n for n in lengths], slots=slots)
        want, at = torch.zeros(total, channels, dtype=torch.float64), 0
        for s, n in enumerate(counts):
            S = want_state[s]
            for t in range(at, at + n):
                S = torch.exp(dt[t].double()[:, None] * A) * S + (dt[t] * x[t]).double()[:, None] * B[t].double()
                zt = z[t].double()
                want[t] = ((S * C[t, :state].double()).sum(1) + D.double() * x[t].double()) * zt * torch.sigmoid(zt)
            want_state[s], at = S, at + n
        out = torch.full((total, channels + 6), float("nan"), device=DEV)
        carry = K.scan_carry(step, channels * state, channels, K.SELECTIVE_SPAN) if spans else None
        on = lambda v: v.contiguous().to(DEV)
        bc = on(torch.cat([B, C], 1))
        K.selective_scan(on(x), on(z), on(dt), bc[:, :state], bc[:, state:2 * state], A_log.to(DEV), D.to(DEV), out, held, step, carry=carry,
                         span=K.SELECTIVE_SPAN)
        assert bool((out[:, channels:] == 0).all())
        # an exponential and a handful of roundings a token, of decays that sum to at most 1 / (1 - decay) tokens' worth
        assert rel_err(out[:, :channels].cpu(), want) < 3e-6
        for slot, w in zip(slots, want_state):
            assert rel_err(held[slot, :channels * state].view(channels, state).cpu(), w) < 3e-6


# which sequences the scan with eight lanes a channel cuts into spans (only then does it write the room for them): 64 tokens and
# 128 for each wave a SIMD has (four to each of 256 compute units), sequences of three spans of 64 whatever the waves
@pytest.mark.parametrize("channels,state,counts,cut", [
    (2048, 24, [64] * 2, True), (2048, 24, [63] * 2, False), (2048, 16, [56] * 3, False), (2048, 32, [48], False), (4096, 24, [64] * 2, False),
    (4096, 24, [128] * 2, True), (2048, 64, [128] * 8, False), (2048, 24, [192] * 8, True), (2048, 24, [200] * 9, False)])
def test_which_sequences_eight_lanes_cut(channels, state, counts, cut):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are those of 256 compute units")
    total = sum(counts)
    step = make_step(torch.float32, counts)
    x, z, dt, bc = [torch.rand(total, n, device=DEV) for n in (channels, channels, channels, 2 * state)]
    A_log, D = torch.zeros(channels, state, device=DEV), torch.zeros(channels, device=DEV)
    held, out = torch.zeros(len(counts), channels * state, device=DEV), torch.empty(total, channels, device=DEV)
    carry = K.scan_carry(step, channels * state, channels, K.SELECTIVE_SPAN)
    if carry is None:
        assert not cut
        return
    carry.fill_(float("nan"))
    K.selective_scan(x, z, dt, bc[:, :state], bc[:, state:], A_log, D, out, held, step, carry=carry, span=K.SELECTIVE_SPAN)
    assert bool(torch.isfinite(carry).any()) == cut
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(held).all())


# a long sequence is cut into spans whatever stands beside it: single tokens are no waves that would fill the chip
@pytest.mark.parametrize("channels,state,counts,cut", [
    (2048, 16, [1000] + [1] * 32, True), (2048, 16, [300] * 8, True), (2048, 16, [1000] * 40, False), (2048, 32, [500] + [1] * 63, True),
    (2048, 16, [64] + [1] * 31, False), (4096, 16, [40] + [1] * 63, False)])
def test_which_sequences_lanes_cut(channels, state, counts, cut):
    test_which_sequences_eight_lanes_cut(channels, state, counts, cut)


# which way a step goes (only blocks write their room): the longest sequence, how many are short beside it, sizes of heads and states;
# `spans`: with room for spans
@pytest.mark.parametrize("form,heads,dim,vdim,counts,spans,blocked", [
    ("head", 8, 128, 128, [1024] * 2, False, True), ("head", 8, 128, 128, [39], False, False), ("channel", 8, 128, 128, [40], False, True),
    ("head", 8, 128, 128, [40] + [1] * 63, False, False), ("head", 8, 128, 128, [500] + [1] * 63, False, True), ("head", 2, 16, 16, [40], False, False),
    ("forget", 8, 128, 128, [100] * 16, True, True), ("forget", 2, 16, 16, [1000], True, False), ("forget", 2, 16, 16, [1000], False, True),
    ("forget", 8, 128, 128, [4000], True, True), ("scan", 32, 128, 64, [1024] * 2, True, True), ("scan", 8, 16, 64, [1000], True, False),
    ("scan", 32, 128, 64, [64] + [1] * 31, True, False), ("scan", 32, 128, 64, [300] + [1] * 20, True, True)])
def test_which_steps_go_in_blocks(form, heads, dim, vdim, counts, spans, blocked):
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are those of 256 compute units")
    gen, total, inner = torch.Generator().manual_seed(9), sum(counts), heads * vdim
    step = make_step(torch.float32, counts)
    state, y = torch.zeros(len(counts), heads * dim * vdim, device=DEV), torch.empty(total, inner, device=DEV)
    if form == "scan":
        room, carry = K.head_blocks(step, heads, vdim, dim, 1), K.scan_carry(step, heads * dim * vdim, heads) if spans else None
        on, zeros = torch.randn(total, inner + 2 * dim + heads, generator=gen).to(DEV), torch.zeros(heads, device=DEV)
    else:
        qk, decays = heads * dim, heads if form == "head" else heads * dim
        room, carry = K.scan_blocks(step, heads, dim, vdim), K.scan_carry(step, heads * dim * vdim, heads * dim) if spans else None
        on, zeros = torch.randn(total, 2 * qk + inner + decays + heads, generator=gen).to(DEV), torch.zeros(decays, device=DEV)
    room.fill_(float("nan"))
    if form == "scan":
        K.head_scan(on[:, :inner], on[:, inner:inner + dim], on[:, inner + dim:inner + 2 * dim], on[:, inner + 2 * dim:], zeros, zeros, zeros, y, state,
                    step, heads, vdim, dim, 1, carry=carry, blocks=room)
    else:
        extra = dict(g_bias=zeros, lower=zeros + 0.5) if form == "forget" else \
            dict(beta=on[:, -heads:], A_log=zeros[:heads], unit=True, q_scale=dim ** -0.5, decay_per_head=form == "head", dt_bias=zeros)
        K.keyed_scan(on[:, :qk], None if form == "forget" else on[:, qk:2 * qk], on[:, 2 * qk:2 * qk + inner], on[:, 2 * qk + inner:2 * qk + inner + decays],
                     y, state, step, heads, heads, dim, vdim, "forget" if form == "forget" else "delta", carry=carry, blocks=room, **extra)
    assert bool(torch.isfinite(room).any()) == blocked
    assert bool(torch.isfinite(y).all()) and bool(torch.isfinite(state).all())


def test_steep_decays_of_channels_in_lanes():
    """A decay's exponent is the step times exp(A_log), however large that is: steps of nearly nothing, of nothing and without end."""
    gen, channels, state, total = torch.Generator().manual_seed(10), 70, 16, 100
    A_log = torch.rand(channels, state, generator=gen) * 2.0
    A_log[::3] = torch.rand(A_log[::3].shape, generator=gen) * 3.0 + 18.0          # exp(A_log): 6.6e7 to 1.3e9
    A_log[5] = 80.0
    x, z, B, C = [torch.randn(total, n, generator=gen) for n in (channels, channels, state, state)]
    dt = torch.exp(torch.rand(total, channels, generator=gen) * 4.0 - 21.0)          # 7.6e-10 to 4e-8
    dt[40, ::2], dt[41], x[41], dt[60, 5] = 0.0, float("inf"), 0.0, 1e-30
    x[40] = x[60] = 0.0
    S, want = torch.zeros(channels, state, dtype=torch.float64), []
    A = -torch.exp(A_log.double())
    for t in range(total):
        step = dt[t].double()[:, None]
        S = torch.exp((step * A).clamp(min=-800.0)) * S + torch.where(x[t][:, None] == 0, 0.0, step * x[t].double()[:, None] * B[t].double())
        zt = z[t].double()
        want.append((S * C[t].double()).sum(1) * zt * torch.sigmoid(zt))
    held, out = torch.zeros(1, channels * state, device=DEV), torch.empty(total, channels, device=DEV)
    step = make_step(torch.float32, [total])
    dt[41] = 1e38                                                       # (an infinite step times no input is not a number)
    on = lambda v: v.contiguous().to(DEV)
    bc = on(torch.cat([B, C], 1))
    K.selective_scan(on(x), on(z), on(dt), bc[:, :state], bc[:, state:], on(A_log), torch.zeros(channels, device=DEV), out, held, step,
                     carry=K.scan_carry(step, channels * state, channels, K.SELECTIVE_SPAN), span=K.SELECTIVE_SPAN)
    # exponents of up to 50 are products rounded to 32 bits: 50 * 2^-24, a few tokens' worth
    assert rel_err(out.cpu(), torch.stack(want)) < 1e-5
    assert rel_err(held.view(channels, state).cpu(), S) < 1e-5
