"""Few-row products whose workgroups take pairs of low tiles of the matrix's rows (csrc/gemm_bf16.hip: tiles_per_workgroup),
at the widths around a round of the chip, against float32 products of the same operands."""
import pytest
import torch

import util

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# in rows per compute unit: one round of single tiles, just over it, pairs of every height, two rounds of pairs
PER_UNIT = (16, 16.03, 17, 18, 20, 21.97, 22, 23.5, 24, 26, 36, 40)


def _width(per_unit, step=8):
    units = torch.cuda.get_device_properties(0).multi_processor_count
    return -(-int(per_unit * units) // step) * step


def _close(got, want, K, rounded):
    """Sums of K products of bfloat16 operands in float32: each within K 2^-24 of the sum of magnitudes, here below
    2^-10 of the largest; results rounded to bfloat16 2^-9 beside it."""
    assert torch.isfinite(got).all()
    assert util.rel_err(got, want) < 2 ** -10 + (2 ** -8 if rounded else 0)


@pytest.mark.parametrize("M", [2, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("per_unit", PER_UNIT)
def test_plain_products(per_unit, M):
    from gpt_fast_amd.ops import gemm_bf16 as G
    N, K = _width(per_unit), 520
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    want = x.float() @ w.float().t()
    _close(G.skinny(x, w, out_dtype=torch.float32), want, K, False)
    _close(G.skinny(x, w), want, K, True)


@pytest.mark.parametrize("M", [3, 8, 16])
@pytest.mark.parametrize("per_unit", PER_UNIT)
def test_into_the_stream_and_the_norm_behind(per_unit, M):
    from gpt_fast_amd.ops import gemm_bf16 as G
    N, K, eps = _width(per_unit), 264, 1e-5
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    w2 = (torch.randn(256, N, generator=g, device=DEV) * 0.05).bfloat16()
    weight = 1 + 0.1 * torch.randn(N, generator=g, device=DEV)
    residual = torch.randn(M, N, generator=g, device=DEV)
    stream = residual + x.float() @ w.float().t()
    xg, ssq = G.skinny_into_chain(x, w, residual, weight)
    _close(residual, stream, K, False)
    want = ((stream * weight).bfloat16().double() * (stream.double().square().mean(1, keepdim=True) + eps).rsqrt()) @ w2.double().t()
    _close(G.skinny_after_chain(xg, ssq, eps, w2, out_dtype=torch.float32), want, N, True)    # a row's bfloat16 may fall either way


@pytest.mark.parametrize("heads,kv_heads", [(60, 6), (64, 8), (70, 9), (88, 10)])
@pytest.mark.parametrize("M", [3, 7, 16])
def test_rotation_and_cache_write(heads, kv_heads, M):
    """Heads of 64: 4,608, 5,120, 5,632 and 6,912 rows of q, k and v."""
    from gpt_fast_amd.ops import gemm_bf16 as G
    hd, K, rot = 64, 264, 48
    N = (heads + 2 * kv_heads) * hd
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    freqs = 10000.0 ** (-torch.arange(0, rot, 2, device=DEV).float() / rot)
    pos = (torch.arange(M, device=DEV) * 5 + 3).int()
    seq = torch.zeros(M, dtype=torch.int32, device=DEV)
    table = torch.tensor([[2, 0]], dtype=torch.int32, device=DEV)
    k_pages = torch.zeros(3, kv_heads, 64, hd, dtype=torch.bfloat16, device=DEV)
    v_pages = torch.zeros(3, kv_heads, hd, 64, dtype=torch.bfloat16, device=DEV)
    q = G.qkv_rope_store(x, w, freqs, seq, pos, table, k_pages, v_pages, heads, kv_heads, hd, rot)
    plain = (x.float() @ w.float().t()).view(M, heads + 2 * kv_heads, hd)
    pairs = plain[:, :heads + kv_heads, :rot].unflatten(-1, (-1, 2)).double()
    angle = (pos[:, None].float() * freqs).double()[:, None]
    a, b = pairs.unbind(-1)
    turned = torch.stack([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1).flatten(-2)
    want = plain.double()
    want[:, :heads + kv_heads, :rot] = turned
    _close(q.view(M, heads, hd), want[:, :heads], K, True)
    keys, values = util.from_cache_order(k_pages, v_pages)
    for m in range(M):
        p = int(pos[m])
        page = int(table[0, p // 64])
        _close(keys[page, :, p % 64], want[m, heads:heads + kv_heads], K, True)
        _close(values[page, :, :, p % 64], want[m, heads + kv_heads:], K, True)


# pairs are a matter of long columns where the rows of x are few: (rows of x, columns of W) on both sides of each line
LINES = [(2, 4096), (4, 4096), (4, 4088), (5, 3072), (8, 3064), (9, 2048), (12, 2040), (13, 64), (9, 4096), (10, 4088), (10, 4096)]


def _within(got, want, x, w, rounded):
    """Sums of K products in float32, in any order: within K 2^-24 of the sum of their magnitudes."""
    bound = x.shape[1] * 2 ** -24 * (x.float().abs() @ w.float().abs().t()) + (2 ** -8 * want.abs() if rounded else 0)
    assert bool(((got.double() - want.double()).abs() <= bound).all())


@pytest.mark.parametrize("per_unit", [17, 19.5, 20, 21.5, 23.5])
@pytest.mark.parametrize("M,K", LINES)
def test_both_sides_of_every_line(M, K, per_unit):
    from gpt_fast_amd.ops import gemm_bf16 as G
    N = _width(per_unit, 64)
    g = torch.Generator(device=DEV).manual_seed(N + M)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    want = x.float() @ w.float().t()
    _within(G.skinny(x, w, out_dtype=torch.float32), want, x, w, False)
    residual, weight = torch.randn(M, N, generator=g, device=DEV), 1 + 0.1 * torch.randn(N, generator=g, device=DEV)
    stream = residual + want
    xg, ssq = G.skinny_into_chain(x, w, residual, weight)
    _within(residual, stream, x, w, True)
    assert util.rel_err(ssq.sum(0)[:M], stream.square().sum(1)) < 2 ** -10
    hd, kv_heads = 64, 4
    heads = N // hd - 2 * kv_heads
    pos = (torch.arange(M, device=DEV) * 5 + 3).int()
    seq = torch.zeros(M, dtype=torch.int32, device=DEV)
    table = torch.tensor([[2, 0]], dtype=torch.int32, device=DEV)
    k_pages = torch.zeros(3, kv_heads, 64, hd, dtype=torch.bfloat16, device=DEV)
    v_pages = torch.zeros(3, kv_heads, hd, 64, dtype=torch.bfloat16, device=DEV)
    freqs = torch.zeros(hd // 2, device=DEV)                          # no turn: the projection itself
    q = G.qkv_rope_store(x, w, freqs, seq, pos, table, k_pages, v_pages, heads, kv_heads, hd, hd)
    _within(q.view(M, -1), want[:, :heads * hd], x, w[:heads * hd], True)
    keys, values = util.from_cache_order(k_pages, v_pages)
    at = (table[0, pos.long() // 64].long(), pos.long() % 64)
    got = torch.cat([keys[at[0], :, at[1]].reshape(M, -1), values[at[0], :, :, at[1]].reshape(M, -1)], 1)
    _within(got, want[:, heads * hd:], x, w[heads * hd:], True)


def test_where_pairs_begin():
    """One workgroup a tile of at least twelve rows of W, or a pair: fewer than a round of the chip."""
    import ctypes
    from gpt_fast_amd.ops.library import library
    units = torch.cuda.get_device_properties(0).multi_processor_count
    workgroups, i = library("gemm_bf16").gfa_skinny_workgroups, ctypes.c_int

    def pairs(mode, M, K, per_unit):
        return workgroups(i(mode), i(M), i(_width(per_unit)), i(K)) <= units
    for M, K in ((4, 4096), (8, 3072), (12, 2048), (16, 8)):
        assert pairs(0, M, K, 18) and pairs(2, M, K, 18) and (M > 8 or not pairs(0, M, K, 24.1))
        assert K == 8 or not pairs(0, M, K - 8, 18)
    assert not pairs(0, 4, 4096, 20.5) and pairs(0, 5, 4096, 20.5)
    assert pairs(4, 10, 4096, 18) and not pairs(4, 9, 4096, 18) and not pairs(4, 16, 4088, 18)
