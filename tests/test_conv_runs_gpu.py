"""The causal convolution of steps of many tokens, which takes runs of tokens, against float64."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K

from step_helpers import make_step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# runs that begin a sequence, straddle two or three (down to one token), end with the step; taps that have runs and one
# that has not; channels that do not fill a work-group; the products' type beside, with columns behind the channels
@pytest.mark.parametrize("taps", [2, 3, 4, 5])
@pytest.mark.parametrize("lengths,channels,act,dtype", [([384], 40, "silu", None), ([3, 1, 2, 400, 9, 17], 300, "none", "bfloat16"),
                                                        ([64] * 7, 257, "silu", "float32"), ([390], 900, "silu", None), ([3, 1, 2, 400, 9, 17], 1000, "none", "bfloat16"),
                                                        ([1] * 20 + [380] + [5] * 9, 900, "silu", "float32"),
                                                        ([3, 1, 2, 400, 9, 17], 2400, "none", "bfloat16"), ([1] * 20 + [380] + [5] * 9, 2300, "silu", "float32")])
def test_runs_of_tokens(taps, lengths, channels, act, dtype):
    gen = torch.Generator().manual_seed(taps * 100 + channels)
    weight, bias = torch.randn(channels, taps, generator=gen), torch.randn(channels, generator=gen)
    slots = list(reversed(range(len(lengths))))
    state = torch.randn(len(lengths), (taps - 1) * channels + 3, generator=gen)
    held = state.to(DEV)
    past = [state[slot, :(taps - 1) * channels].view(taps - 1, channels).double() for slot in slots]
    for part in range(2):
        rows = torch.randn(sum(lengths), channels + 5, generator=gen)
        step = make_step(torch.float32, lengths, starts=[part * n for n in lengths], slots=slots)
        out = torch.full((sum(lengths), channels + 2), float("nan"), device=DEV)
        cast = torch.full((sum(lengths), channels + 8), float("nan"), dtype=getattr(torch, dtype), device=DEV) if dtype else None
        K.causal_conv(rows.to(DEV)[:, :channels], weight.to(DEV), bias.to(DEV), out, held, step, cast=cast, act=act)
        at = 0
        for s, n in enumerate(lengths):
            u = torch.cat([past[s], rows[at:at + n, :channels].double()])
            want = bias.double() + sum(u[j:j + n] * weight[:, j].double() for j in range(taps))
            want = want * torch.sigmoid(want) if act == "silu" else want
            got = out[at:at + n, :channels].cpu().double()
            # a handful of 32-bit roundings of values of size one to ten
            assert float((got - want).abs().max()) < 5e-6
            if dtype:
                assert torch.equal(cast[at:at + n, :channels].cpu(), out[at:at + n, :channels].cpu().to(cast.dtype))
            past[s] = u[n:]
            assert torch.equal(held[slots[s], :(taps - 1) * channels].view(taps - 1, channels).cpu().double(), past[s])
            at += n
        assert bool(torch.isnan(out[:, channels:]).all()) and (cast is None or bool((cast[:, channels:] == 0).all()))
