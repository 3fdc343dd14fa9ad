"""The tile kernel's forms on blocks of 16 x 16: counts of tiles of K around their stages, ragged edges, every epilogue, keys and
values scattered (quads of positions together, quads that start inside one, rows of two sequences in a quad)."""

import pytest
import torch

import test_tile_forms_gpu as forms

pytestmark = pytest.mark.gpu
BLOCK_FORMS = (2, 3) + tuple(range(6, 15))


@pytest.fixture(autouse=True)
def block_forms(monkeypatch):
    monkeypatch.setitem(forms.FORMS, torch.bfloat16, BLOCK_FORMS)


# (two to eight stages; tiles of 64 to 256 rows and 64 to 256 columns)
@pytest.mark.parametrize("m,n,tiles", [(65, 64, 1), (128, 256, 2), (130, 136, 3), (257, 264, 4), (300, 129, 5), (70, 514, 7), (258, 104, 9), (513, 328, 24)])
def test_epilogues(m, n, tiles):
    forms.test_epilogues_of_every_form(torch.bfloat16, m, n, tiles)


@pytest.mark.parametrize("heads,kv_heads,hd", [(4, 4, 64), (3, 1, 128), (4, 2, 32), (5, 5, 48), (2, 2, 80), (3, 3, 16)])
def test_scattered(heads, kv_heads, hd):
    forms.test_scattered_keys_and_values(torch.bfloat16, heads, kv_heads, hd)
