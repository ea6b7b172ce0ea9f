"""One plain layer over a few rows (csrc/resident_layers.hip, and beside it the launches of one kernel at a time,
csrc/gemm_bf16.hip: gfa_few_row_layers_bf16), row by row, with the keys and values that it writes."""
from types import SimpleNamespace

import pytest
import torch

import util

pytestmark = pytest.mark.gpu
DEV, PAGE, EPS = "cuda:0", 64, 1e-5


def _problem(D, H, G, hd, inner, held, new, window=0, rot=None, seed=0, extra_pages=0):
    """A layer, its inputs and a cache that holds ``held`` tokens of each sequence; slots that hold none are NaN."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def randn(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device=DEV) * std
    rot = hd if rot is None else rot
    M, longest = sum(new), max(h + n for h, n in zip(held, new))
    width = -(-longest // PAGE) + extra_pages
    n_pages = width * len(held) + 2
    table = torch.randperm(n_pages, generator=g, device=DEV)[:width * len(held)].view(len(held), width).int()
    keys = torch.full((n_pages, G, PAGE, hd), float("nan"), device=DEV, dtype=torch.bfloat16)
    values = torch.full((n_pages, G, hd, PAGE), float("nan"), device=DEV, dtype=torch.bfloat16)
    for i, h in enumerate(held):
        for at in range(0, h, PAGE):
            n, page = min(PAGE, h - at), int(table[i, at // PAGE])
            keys[page, :, :n] = randn(G, n, hd).bfloat16()
            values[page, :, :, :n] = randn(G, hd, n).bfloat16()
    p = SimpleNamespace(
        D=D, H=H, G=G, hd=hd, inner=inner, rot=rot, window=window, scale=hd ** -0.5, held=held, new=new, keys=keys, values=values,
        wqkv=randn((H + 2 * G) * hd, D, std=D ** -0.5).bfloat16(), wo=randn(D, H * hd, std=(H * hd) ** -0.5).bfloat16(),
        w13=randn(2 * inner, D, std=D ** -0.5).bfloat16(), w2=randn(D, inner, std=inner ** -0.5).bfloat16(),
        norm_mixer=1 + 0.1 * randn(D), norm_ffn=1 + 0.1 * randn(D), table=table, residual=randn(M, D),
        freqs=10000.0 ** (-torch.arange(0, rot, 2, device=DEV).float() / rot))
    ints = dict(dtype=torch.int32, device=DEV)
    starts = [sum(new[:i]) for i in range(len(new) + 1)]
    p.batch = SimpleNamespace(
        tok_seq=torch.tensor([i for i, n in enumerate(new) for _ in range(n)], **ints),
        tok_pos=torch.tensor([h + t for h, n in zip(held, new) for t in range(n)], **ints),
        start_pos=torch.tensor(held, **ints), q_start=torch.tensor(starts, **ints), n_seqs=len(new), n_tokens=M, max_q_len=max(new))
    return p


def _layer(p):
    """The layer with a cache of its own in the kernels' order."""
    from gpt_fast_amd.ops import few_row_layers as F
    return F.Layer(p.wqkv, p.wo, p.w13, p.w2, p.norm_mixer, p.norm_ffn, *util.to_cache_order(p.keys, p.values), p.table)


def _resident(p, layers, stream, **options):
    from gpt_fast_amd.ops import resident_layers as R
    R.run(layers, stream, p.freqs, p.rot, p.batch, p.H, p.G, p.hd, p.window, EPS, EPS, p.scale, "silu", **options)


def _run(p, way, **options):
    """(the stream behind the layer, its keys and values as [page, G, slot, d] and [page, G, d, slot])."""
    from gpt_fast_amd.ops import few_row_layers as F
    layer, stream = _layer(p), p.residual.clone()
    if way == "resident":
        _resident(p, [layer], stream, **options)
    else:
        x = stream * (stream.square().mean(1, keepdim=True) + EPS).rsqrt() * p.norm_mixer
        F.run_layers([layer], x.bfloat16(), stream, p.freqs, p.rot, p.batch, p.H, p.G, p.hd, p.window, EPS, EPS, p.scale, "silu")
    return (stream,) + util.from_cache_order(layer.k_pages, layer.v_pages)


# head size, heads, key/value heads, window, the newest token's position; the keys that are no numbers: all that a wave sees, the
# first time the only one of its block of 32 that the window shows, the last time all of a share of a long context
NO_NUMBERS = [(64, 4, 4, 65, 95, 31, 32), (128, 8, 2, 0, 70, 32, 64), (48, 6, 3, 0, 40, 0, 32), (16, 2, 2, 0, 96, 64, 96),
              (64, 2, 1, 0, 2100, 0, 256)]


@pytest.mark.parametrize("way", ["resident", "one by one"])
@pytest.mark.parametrize("hd,H,G,window,pos,first,end", NO_NUMBERS)
def test_a_part_of_a_context_that_is_no_number_makes_the_row_no_number(hd, H, G, window, pos, first, end, way):
    """Every column of the layer's result reads every head, so the row is NaN from end to end; the other sequence's row keeps
    its bits."""
    p = _problem(128, H, G, hd, 136, [pos, pos], [1, 1], window=window)
    want = _run(p, way)[0]
    assert bool(torch.isfinite(want).all())
    for key in range(first, end):
        p.keys[int(p.table[0, key // PAGE]), :, key % PAGE] = float("nan")
    got = _run(p, way)[0]
    assert bool(torch.isnan(got[0]).all())
    assert torch.equal(got[1], want[1])


# width, heads, key/value heads, head size, inner; held tokens, new ones; window, dims turned.  Rows kept: 1, 2, 4, 8, 16.  x of a
# product whole, and in halves: of the columns of a streamer 20 128-wide pieces of 49 at a time (one row of 49,160), 10 of 28 (two
# rows of 28,672), 5 of 14 (four of 14,336), 2 of 11 (eight of 11,008), 2 of 8 (eight of 64 heads of 128), 1 of 3 (twelve of 3,072)
ROW_BY_ROW = [(768, 12, 12, 64, 2048, [700, 40], [1, 1], 0, 64), (768, 12, 4, 64, 2048, [0], [4], 0, 64),
              (128, 2, 1, 64, 49160, [33], [1], 0, 64), (256, 4, 2, 64, 28672, [90, 3], [1, 1], 0, 64),
              (256, 4, 2, 64, 14336, [5, 6, 700], [1, 1, 1], 0, 64), (256, 4, 2, 64, 14336, [20], [4], 0, 64),
              (264, 4, 4, 64, 11008, [9] * 5 + [2100], [1] * 5 + [3], 0, 64), (256, 64, 8, 128, 520, [70] * 8, [1] * 8, 0, 128),
              (3072, 4, 1, 128, 136, [3] * 12, [1] * 12, 0, 128), (1032, 16, 2, 48, 1104, [2100] + [31] * 15, [1] * 16, 0, 48),
              (200, 10, 5, 80, 328, [700, 31, 64], [1, 2, 3], 70, 30), (128, 16, 1, 128, 264, [0], [16], 0, 2)]


def _exact(p):
    """The layer in 64 bits: (the stream behind it, the new tokens' keys and values [M, G, hd])."""
    f, hd, G = torch.float64, p.hd, p.G

    def normed(x, weight):
        return x * (x.square().mean(1, keepdim=True) + EPS).rsqrt() * weight.to(f)
    stream, pos, seq = p.residual.to(f), p.batch.tok_pos.long(), p.batch.tok_seq.long()
    M = len(pos)
    q, k, v = (normed(stream, p.norm_mixer) @ p.wqkv.to(f).t()).view(M, -1, hd).split([p.H, G, G], 1)
    angle = (pos[:, None].float() * p.freqs).to(f)[:, None]

    def turned(x):
        a, b = x[..., :p.rot].unflatten(-1, (-1, 2)).unbind(-1)
        pair = torch.stack([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)
        return torch.cat([pair.flatten(-2), x[..., p.rot:]], -1)
    q, k = turned(q), turned(k)
    mixed = torch.empty_like(q)
    for t in range(M):
        at = torch.arange(max(0, int(pos[t]) + 1 - p.window) if p.window else 0, int(pos[t]) + 1, device=DEV)
        page, slot = p.table[seq[t]].long()[at // PAGE], at % PAGE
        keys, values = p.keys[page, :, slot].to(f), p.values[page, :, :, slot].to(f)          # [keys, G, hd]
        for i in range(M):                                                # those of this step, as they were written
            if seq[i] == seq[t] and at[0] <= pos[i] <= pos[t]:
                keys[pos[i] - at[0]], values[pos[i] - at[0]] = k[i], v[i]
        rows = q[t].view(G, -1, hd)
        for g in range(G):
            mixed[t].view(G, -1, hd)[g] = (rows[g] @ keys[:, g].t() * p.scale).softmax(-1) @ values[:, g]
    stream = stream + mixed.reshape(M, -1) @ p.wo.to(f).t()
    a, b = (normed(stream, p.norm_ffn) @ p.w13.to(f).t()).chunk(2, 1)
    return stream + (torch.nn.functional.silu(a) * b) @ p.w2.to(f).t(), k, v


@pytest.mark.parametrize("workgroups", [0, 7])
@pytest.mark.parametrize("sizes", ROW_BY_ROW, ids=str)
def test_every_row_and_what_it_leaves_in_the_cache(sizes, workgroups):
    """Against 64 bits, each row by itself.  bfloat16 rounds by at most 2^-9 of a value: a key or a value through the norm's rows and
    its own rounding, 2^-8 of the row at most beside sums in float32; what the layer adds to the stream through seven such roundings one
    behind the other (rows, queries, probabilities, heads, rows, gate; keys and values beside them), independent of
    one another, sqrt(7) 2^-9 < 2^-7.  A 128-wide piece left out of 14,336 columns changes a row by a tenth."""
    D, H, G, hd, inner, held, new, window, rot = sizes
    p = _problem(D, H, G, hd, inner, held, new, window=window, rot=rot, seed=3)
    want, k, v = _exact(p)
    stream, keys, values = _run(p, "resident", workgroups=workgroups)
    at = p.batch.tok_pos.long()
    page, slot = p.table[p.batch.tok_seq.long(), at // PAGE].long(), at % PAGE
    for name, got, right, bound in (("stream", stream - p.residual, want - p.residual, 2 ** -7),
                                    ("keys", keys[page, :, slot], k, 2 ** -8), ("values", values[page, :, :, slot], v, 2 ** -8)):
        error = (got.double() - right).flatten(1).norm(dim=1) / right.flatten(1).norm(dim=1)
        print(f"{name}: largest {float(error.max()):.5f} of {bound:.5f}", flush=True)
        assert bool((error <= bound).all()), (name, error)           # false for NaN
    held_still = torch.ones(keys.shape[0], PAGE, dtype=torch.bool, device=DEV)
    held_still[page, slot] = False                                    # nothing else of the cache is written
    for now, was in ((keys, p.keys), (values.transpose(2, 3), p.values.transpose(2, 3))):
        now, was = now.transpose(1, 2)[held_still], was.transpose(1, 2)[held_still]
        assert torch.equal(now.view(torch.int16), was.view(torch.int16))


def test_repeats_have_the_same_bits():
    """Every launch reads what its own workgroups left, also where several of them wrote parts of one line."""
    for sizes in ((768, 12, 12, 64, 2048, [40], [1]), (264, 4, 2, 64, 1096, [9, 300, 70], [1, 1, 1])):
        p = _problem(*sizes)
        layers = [_layer(p) for _ in range(32)]
        results = []
        for _ in range(40):
            stream = p.residual.clone()
            _resident(p, layers, stream)
            results.append(stream)
        assert bool(torch.isfinite(results[0]).all())
        assert all(torch.equal(r, results[0]) for r in results)


def test_a_launch_that_begins_on_a_busy_chip_has_the_rest_of_it_once_it_is_free():
    """32 layers of 4,096 beside two, then four, launches of as many that leave them eight compute units: they
    stay with the eight for a layer, not to their end, which would take 32 times as long as on the whole chip; and what they
    compute has the same bits."""
    p = _problem(4096, 32, 8, 128, 14336, [200, 31], [1, 1])
    units = torch.cuda.get_device_properties(0).multi_processor_count
    mine_layers, other_layers = ([_layer(p) for _ in range(32)] for _ in range(2))      # one set of weights, a cache each
    mine, others = torch.cuda.Stream(), torch.cuda.Stream()
    other_rows = p.residual.clone()

    def timed(**options):
        stream = p.residual.clone()
        torch.cuda.synchronize()
        begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        for _ in range(options.pop("beside", 0)):
            with torch.cuda.stream(others):
                _resident(p, other_layers, other_rows, workgroups=units - 8)
        with torch.cuda.stream(mine):
            begin.record()
            _resident(p, mine_layers, stream, **options)
            end.record()
        torch.cuda.synchronize()
        return stream, begin.elapsed_time(end)
    timed()
    want, alone = timed()
    assert bool(torch.isfinite(want).all())
    for beside in (2, 4):
        got, took = timed(beside=beside, start_polls=1)
        print(f"alone {alone:.2f} ms, beside {beside} launches {took:.2f} ms", flush=True)
        assert torch.equal(got, want)
        assert took < 8 * alone


def test_the_work_memory_holds_the_partial_sums_of_one_layer():
    """8B shape, 8 rows: 32 layers' rows and one set of partial sums, which 64 pages of table allow two a compute unit of."""
    import ctypes
    from gpt_fast_amd.ops.library import library
    size = library("resident_layers").gfa_resident_work_bytes
    size.restype = ctypes.c_long
    units = torch.cuda.get_device_properties(0).multi_processor_count
    sizes = [size(n, 8, 4096, 14336, 32, 8, 128, 64) for n in (1, 2, 32)]
    assert sizes[2] - sizes[1] == 30 * (sizes[1] - sizes[0])
    partials = 2 * max(units, 64) * 4 * (128 + 2) * 4
    rows = 8 * (2 * (3 * 4096 + 2 * 4096 + 14336) + 2 * 4096)         # x of four products, q, shares of the squares at one for four
    assert sizes[1] - sizes[0] < 1.1 * rows and sizes[0] < 1.1 * (rows + partials) + 65536
