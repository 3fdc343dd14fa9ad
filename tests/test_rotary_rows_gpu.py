"""Head norms and rotation into the cache in steps of many tokens."""

import pytest
import torch

from burn_transformers_amd.kernels import library as K
from kernel_helpers import PagedCase

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def rel_err(got, want):
    got = got.detach().cpu().double()
    return float((got - want).abs().max() / want.abs().max().clamp_min(1e-30))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
# tokens on both sides of the rule that chooses the kernel by the heads of all tokens
@pytest.mark.parametrize("longest", [600, 2300])
# heads and sizes on both sides of a wave's four heads and 128 channels, one odd size that the general kernel takes
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,rot,norm,neighbours,same", [
    (8, 2, 128, 128, 64, "head", False, False), (6, 3, 64, 32, 64, "whole", False, False), (2, 1, 128, 128, 128, None, False, False),
    (5, 5, 16, 48, 8, "head", True, False), (4, 4, 32, 32, 0, "whole", False, True), (1, 1, 6, 2, 2, "head", True, False),
    (3, 1, 10, 10, 6, "head", False, False)])
def test_rotation_of_many_tokens(dtype, longest, heads, kv_heads, dim, vdim, rot, norm, neighbours, same):
    dt = DTYPES[dtype]
    hd = (max(dim, vdim) + 15) // 16 * 16
    totals, counts = [longest, 70, 131], [longest, 66, 103]
    case = PagedCase(totals, counts, kv_heads, hd, dt, DEV, seed=1)
    gen = torch.Generator().manual_seed(2)
    n = case.n_tokens
    fused = torch.randn(n, (heads + kv_heads) * dim + (0 if same else kv_heads * vdim), generator=gen)
    spread = 1 if norm != "whole" else None
    q_gamma = torch.randn((spread or heads) * dim, generator=gen) + 1.0
    k_gamma = torch.randn((spread or kv_heads) * dim, generator=gen) + 1.0
    inv_freq = (1000.0 ** (-2.0 * torch.arange(rot // 2, dtype=torch.float64) / max(rot, 1))).float()
    q_out = torch.full((n, heads * hd), float("nan"), dtype=dt, device=DEV)
    K.head_rotary(fused.to(DEV), heads, kv_heads, dim, vdim, rot, inv_freq.to(DEV) if rot else None, q_gamma.to(DEV) if norm else None,
                  k_gamma.to(DEV) if norm else None, 1e-3, q_out, case.tok_seq, case.tok_pos, case.view(), dt, neighbours=neighbours,
                  whole_norm=norm == "whole", amplitude=1.25, values_from_keys=same, temperature=(0.1, 64))
    pos = case.tok_pos.cpu().double()

    def heads_of(first, count, size, gamma):
        rows = fused.double()[:, first:first + count * size].reshape(n, count, size)
        if gamma is not None and norm:
            squares = (rows * rows).mean((1, 2) if norm == "whole" else -1, keepdim=True)
            rows = rows / torch.sqrt(squares + 1e-3) * gamma.double().reshape(-1, size)
        if gamma is not None and rot:
            angle = (pos[:, None].float() * inv_freq[None]).double()             # the angle itself is a 32-bit product
            cos, sin = 1.25 * torch.cos(angle)[:, None], 1.25 * torch.sin(angle)[:, None]
            half = rot // 2
            at = torch.arange(half)
            one, two = (2 * at, 2 * at + 1) if neighbours else (at, at + half)
            turned = rows.clone()
            turned[..., one] = rows[..., one] * cos - rows[..., two] * sin
            turned[..., two] = rows[..., two] * cos + rows[..., one] * sin
            rows = turned
        out = torch.zeros(n, count, hd, dtype=torch.float64)
        out[..., :size] = rows
        return out.reshape(n, count * hd)

    # float32: the angle's product is the same, a dozen roundings of 2^-24 follow; bfloat16: half a unit of the largest, 2^-9
    bound = 2e-6 if dtype == "float32" else 2.0 ** -8
    factor = 1.0 + 0.1 * torch.log(torch.floor((pos + 1) / 64) + 1.0)
    assert rel_err(q_out, heads_of(0, heads, dim, q_gamma) * factor[:, None]) < bound
    k_all, v_all = case.read_back()
    rows, at = [], 0
    for total, count in zip(totals, counts):
        rows += list(range(at + total - count, at + total))
        at += total
    assert rel_err(k_all[rows], heads_of(heads * dim, kv_heads, dim, k_gamma)) < bound
    assert rel_err(v_all[rows], heads_of((heads + (0 if same else kv_heads)) * dim, kv_heads, vdim, None)) < bound

