"""The experts' tile kernel where its rings of buffers begin and end."""
import pytest
import torch

from util import rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tile", [1, 2, 4])
@pytest.mark.parametrize("pieces", [1, 2, 3, 4, 5, 6, 7])
def test_fewer_pieces_of_k_than_buffers_and_a_few_more(monkeypatch, tile, pieces):
    """Tiles of every height (one to four steps of 64 rows), columns beyond a whole tile and beyond what an XCD
    takes together, and as many pieces of 64 k as make every number of stages behind the last copy; against the same
    bfloat16 operands in float64.  The result is rounded to bfloat16 once: neighbours lie 2^-7 of their power of two apart
    (eight bits of significand, the leading one among them), so that a value moves by at most half of that, 2^-8 of itself,
    after float32 sums of up to 448 products (2^-24 each)."""
    from gpt_fast_amd.ops import routed_experts as RE
    monkeypatch.setattr(RE, "_tile_of", lambda *a: tile)
    counts, K, F = [60, 0, 128, 190, 256, 257], 64 * pieces, 1288
    g = torch.Generator().manual_seed(pieces)
    x = torch.randn(sum(counts), K, generator=g).bfloat16()
    w = (torch.randn(len(counts), F, K, generator=g) * 0.3).bfloat16()
    offsets = torch.tensor([sum(counts[:i]) for i in range(len(counts) + 1)], dtype=torch.int32)
    got = RE.expert_tile_product(x.to(DEV), None, 1, w.to(DEV), offsets.to(DEV), None, sum(counts)).double().cpu()
    want = torch.cat([x[sum(counts[:e]):sum(counts[:e + 1])].double() @ w[e].double().T for e in range(len(counts))])
    assert rel_err(got, want) < 2.0 ** -8


@pytest.mark.parametrize("activation,gated", [(None, False), ("gelu", False), ("silu", True)])
@pytest.mark.parametrize("pieces", [3, 9, 20])
def test_tiles_of_every_size_give_the_same_bits(monkeypatch, activation, gated, pieces):
    """A row's sums go through K in an order that depends on its expert alone, whichever tile the step's rows asked for:
    columns beyond four tiles of any width, experts whose first pieces differ."""
    from gpt_fast_amd.ops import routed_experts as RE
    counts, K, F = [60, 0, 128, 190, 256, 257], 64 * pieces, 2056
    g = torch.Generator().manual_seed(pieces)
    x = torch.randn(sum(counts), K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(len(counts), 2 * F if gated else F, K, generator=g) * 0.1).bfloat16().to(DEV)
    offsets = torch.tensor([sum(counts[:i]) for i in range(len(counts) + 1)], dtype=torch.int32).to(DEV)
    out = {}
    for tile in (1, 2, 4):
        monkeypatch.setattr(RE, "_tile_of", lambda *a: tile)
        out[tile] = RE.expert_tile_product(x, None, 1, w, offsets, None, sum(counts), activation, gated)
    assert torch.equal(out[1], out[4])
    assert torch.equal(out[2], out[4])
