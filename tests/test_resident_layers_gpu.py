"""Few-row steps through plain layers in one launch (csrc/resident_layers.hip) against the same model in float32, beside
the launches of one kernel at a time (ops/few_row_layers.py), and the rule that chooses between the two."""
import dataclasses

import pytest
import torch

import util

gpu = pytest.mark.gpu

# (hidden, heads, key/value heads, head size, inner, layers): every head size class; widths that are no multiple of 16 or
# of 128; x in one piece, in halves (6008 wide from 8 rows on, 4096 from 16 on); more layers than a launch takes
SHAPES = {"16": (64, 4, 4, 16, 176, 8), "48": (200, 10, 5, 48, 328, 9), "128": (256, 16, 1, 128, 400, 8), "80": (328, 4, 2, 80, 6008, 8),
          "1032": (1032, 12, 12, 64, 1104, 8), "4096": (4096, 4, 1, 64, 40, 8), "33 layers": (128, 2, 1, 64, 264, 33)}
# held tokens, then the tokens of the step: a split context, one far longer than the others, no context, short prompts, both
STEPS = [([2100], [1]), ([31, 64, 5], [1, 1, 1]), ([1300] + [9] * 7, [1] * 8), ([3] * 16, [1] * 16), ([0], [5]), ([40, 0], [1, 9]),
         ([600], [7]), ([0], [16])]


def _engines(shape, monkeypatch, changed=lambda layer: layer):
    """The model in bfloat16 and in float32, of the same weights."""
    import gpt_fast_amd as gfa
    from gpt_fast_amd.weights.random_init import random_parameters
    hidden, heads, kv_heads, head_dim, inner, layers = SHAPES[shape]
    config = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": hidden, "num_hidden_layers": layers,
              "num_attention_heads": heads, "num_key_value_heads": kv_heads, "head_dim": head_dim, "intermediate_size": inner,
              "vocab_size": 320, "max_position_embeddings": 4096, "rope_theta": 10000.0, "rms_norm_eps": 1e-5,
              "rope_scaling": None, "tie_word_embeddings": False}
    arch = gfa.config.registry.architecture_of(config)
    config = arch.read_config(config)
    plan = arch.plan(config)
    plan = dataclasses.replace(plan, layers=[changed(layer) for layer in plan.layers])
    params = random_parameters(arch.bindings(config), 5, "bfloat16", "cuda:0", std=0.05, norm_std=0.1, tie=False)
    exact = {k: v.float() for k, v in params.items()}
    return (gfa.Engine.from_plan(plan, params, "bfloat16", "cuda:0", max_tokens=16384),
            gfa.Engine.from_plan(plan, exact, "float32", "cuda:0", max_tokens=16384))


def _step(engine, held, new):
    import gpt_fast_amd as gfa
    slots = [engine.start_sequence() for _ in held]
    before = [gfa.Entry(s, util.random_tokens(320, n, 7 + i)) for i, (s, n) in enumerate(zip(slots, held)) if n]
    if before:
        engine.step(before)
    out = engine.step([gfa.Entry(s, util.random_tokens(320, n, 50 + i), want=list(range(n)))
                       for i, (s, n) in enumerate(zip(slots, new))])
    for s in slots:
        engine.end_sequence(s)
    return out.double()


def _compare(shape, monkeypatch, changed=lambda layer: layer, steps=STEPS, **options):
    """Both ways round to bfloat16 at the same places, so that their errors against float32 are two draws of one
    size, which is the model's (8 layers of 1032 at this spread of weights: 0.041 one by one): over all steps of a shape no
    more than a quarter above it, in one step (some tens of independent numbers) no more than double."""
    from gpt_fast_amd.ops import resident_layers as R
    engine, exact = _engines(shape, monkeypatch, changed)
    ran, run = [], R.run
    monkeypatch.setattr(R, "run", lambda layers, *a: (ran.append(len(layers)), run(layers, *a, **options))[1])
    errors = torch.zeros(2, dtype=torch.float64)
    for held, new in steps:
        want = _step(exact, held, new)
        here = []
        for resident in (False, True):
            monkeypatch.setattr(R, "pays", lambda *a: resident)
            del ran[:]
            print(shape, held[:2], new[:2], "resident" if resident else "one by one", flush=True)
            got = _step(engine, held, new)
            assert bool(ran) == resident and ran[-1:] == ([SHAPES[shape][5]] if resident else [])
            here.append(((got - want) ** 2).mean() / (want ** 2).mean())
        assert here[1] <= 4 * here[0], (held, new, here)          # false for NaN
        errors += torch.stack(here).cpu()
    assert errors[1] <= 1.25 ** 2 * errors[0], errors


@gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_resident_layers_are_as_close_to_float32_as_single_launches(shape, monkeypatch):
    _compare(shape, monkeypatch)


@gpu
@pytest.mark.parametrize("shape,window,rotary,activation", [("16", 3, 8, "gelu_tanh"), ("128", 70, 64, "silu"),
                                                            ("48", 700, 2, "gelu_tanh"), ("1032", 1, 30, "gelu_tanh")])
def test_with_a_window_a_part_of_the_rotation_and_the_other_gate(shape, window, rotary, activation, monkeypatch):
    def changed(layer):
        position = dataclasses.replace(layer.mixer.position, rotary_dim=rotary)
        return dataclasses.replace(layer, mixer=dataclasses.replace(layer.mixer, window=window, position=position),
                                   feed_forward=dataclasses.replace(layer.feed_forward, activation=activation))
    _compare(shape, monkeypatch, changed)


@gpu
@pytest.mark.parametrize("shape,workgroups,start_polls", [("16", 1, 0), ("128", 7, 0), ("1032", 200, 0), ("48", 0, 1), ("1032", 0, 1)])
def test_with_fewer_workgroups_and_a_list_of_workers_that_closes_early(shape, workgroups, start_polls, monkeypatch):
    _compare(shape, monkeypatch, steps=STEPS[1:6], workgroups=workgroups, start_polls=start_polls)


@gpu
@pytest.mark.parametrize("held,new", [([300] * 8, [1] * 8), ([900], [6])])
def test_a_captured_step_replays_to_the_same_rows(held, new, monkeypatch):
    import gpt_fast_amd as gfa
    from gpt_fast_amd.ops import resident_layers as R
    engine, _ = _engines("1032", monkeypatch)
    ran, run = [], R.run
    monkeypatch.setattr(R, "run", lambda *a: (ran.append(1), run(*a))[1])
    slots = [engine.start_sequence() for _ in held]
    engine.step([gfa.Entry(s, util.random_tokens(320, n, i)) for i, (s, n) in enumerate(zip(slots, held))])
    with torch.no_grad():
        batch = engine.prepare([gfa.Entry(s, util.random_tokens(320, n, 9 + i), want=list(range(n)), key=i)
                                for i, (s, n) in enumerate(zip(slots, new))])
        want = engine.model.forward(batch, engine.cache).clone()
        assert ran == [1]
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = engine.model.forward(batch, engine.cache)
        for _ in range(4):
            got.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want)
            again = engine.model.forward(batch, engine.cache)
            torch.cuda.synchronize()
            assert torch.equal(again, want)


@gpu
def test_steps_on_two_streams_at_once_share_the_chip(monkeypatch):
    """Neither launch waits for workgroups that the other's keep out, and whoever works out a part, it has the same bits."""
    import gpt_fast_amd as gfa
    from gpt_fast_amd.ops import resident_layers as R
    engine, _ = _engines("1032", monkeypatch)
    ran, run = [], R.run
    monkeypatch.setattr(R, "pays", lambda *a: True)
    monkeypatch.setattr(R, "run", lambda *a: (ran.append(1), run(*a))[1])
    slots = [engine.start_sequence() for _ in range(2)]
    engine.step([gfa.Entry(s, util.random_tokens(320, 200, i)) for i, s in enumerate(slots)])
    with torch.no_grad():
        batches = [engine.prepare([gfa.Entry(s, [5 + i], want=[0])]) for i, s in enumerate(slots)]
        want = [engine.model.forward(b, engine.cache) for b in batches]
        torch.cuda.synchronize()
        assert len(ran) == 2 and all(bool(torch.isfinite(rows).all()) for rows in want)
        streams = [torch.cuda.Stream() for _ in batches]
        got = []
        for _ in range(20):
            for batch, stream in zip(batches, streams):
                with torch.cuda.stream(stream):
                    got.append(engine.model.forward(batch, engine.cache))
        torch.cuda.synchronize()
    assert len(ran) == 42
    for i, rows in enumerate(got):
        assert torch.equal(rows, want[i % 2]), i


def test_the_rule():
    from gpt_fast_amd.ops import resident_layers as R
    small, wide = (768, 2048, 12, 12, 64), (4096, 14336, 32, 8, 128)

    def pays(layers, rows, seqs, pages, sizes):
        return R.pays(layers, rows, seqs, pages, *sizes, 256)
    assert pays(12, 1, 1, 1, small) and pays(12, 16, 16, 8, small) and pays(8, 8, 8, 8, wide) and pays(32, 4, 4, 4096, wide)
    assert not pays(7, 1, 1, 1, small)                        # few layers
    assert not pays(32, 9, 9, 8, wide)                        # many wide rows
    assert pays(12, 16, 16, 8, (2048, 5632, 32, 8, 64)) and not pays(12, 16, 16, 8, (2048, 5640, 32, 8, 64))
    assert pays(32, 8, 8, 8, (4096, 11008, 32, 32, 128)) and not pays(40, 8, 8, 8, (5120, 13824, 40, 40, 128))
    assert pays(32, 2, 2, 192, wide) and not pays(32, 2, 2, 193, wide) and pays(32, 2, 1, 193, wide)


def test_what_the_kernel_takes_and_what_begins_where_it_reads():
    from types import SimpleNamespace
    from gpt_fast_amd.ops import resident_layers as R
    assert R.takes(16, 768, 2048, 12, 12, 64, 64) and R.takes(1, 8, 8, 16, 1, 16, 2) and R.takes(1, 8192, 28672, 64, 8, 128, 128)
    for sizes in ((17, 768, 2048, 12, 12, 64, 64), (0, 768, 2048, 12, 12, 64, 64), (1, 764, 2048, 12, 12, 64, 64),
                  (1, 768, 2052, 12, 12, 64, 64), (1, 768, 2048, 12, 12, 72, 64), (1, 768, 2048, 12, 12, 256, 64),
                  (1, 768, 2048, 17, 1, 64, 64), (1, 768, 2048, 12, 12, 64, 0), (1, 16384, 131072, 128, 8, 128, 128)):
        assert not R.takes(*sizes), sizes
    names = ("wqkv", "wo", "w13", "w2", "norm_mixer", "norm_ffn", "k_pages", "v_pages")
    whole = {n: torch.zeros(64) for n in names}
    residual = torch.zeros(64)
    assert R.aligned([SimpleNamespace(**whole)] * 2, residual) and not R.aligned([SimpleNamespace(**whole)], residual[1:])
    for n in names:
        assert not R.aligned([SimpleNamespace(**whole), SimpleNamespace(**{**whole, n: whole[n][1:]})], residual), n


def test_rows_whose_offsets_do_not_fit_into_32_bits_are_not_taken():
    """Sixteen rows of 2^27 - 8 columns are 2^32 - 256 bytes: what lies behind them in a layer's buffers is out of reach."""
    from gpt_fast_amd.ops import resident_layers as R
    assert R.takes(16, 8, (1 << 23) - 8, 8, 1, 16, 2)
    assert not R.takes(16, 8, 1 << 23, 8, 1, 16, 2) and not R.takes(16, 8, (1 << 27) - 8, 8, 1, 16, 2)
    assert not R.takes(16, 8, 8, 1 << 19, 1 << 19, 16, 2)


def test_the_rule_on_long_contexts():
    """Steps that took longer in one launch than in five a layer, and beside each one that did not."""
    from gpt_fast_amd.ops import resident_layers as R

    def pays(rows, keys, sizes, window=0, seqs=None):
        return R.pays(12, rows, seqs or rows, -(-keys // 64), *sizes, 256, window)
    small, heads_of_32 = (768, 2048, 12, 12, 64), (512, 1376, 16, 16, 32)
    assert pays(8, 2000, small) and not pays(8, 4000, small)
    assert pays(16, 900, small) and not pays(16, 1500, small) and not pays(16, 5000, small)
    assert pays(8, 1500, heads_of_32) and not pays(16, 1500, heads_of_32) and not pays(1, 5000, heads_of_32)
    assert not pays(3, 30000, (2048, 5632, 32, 4, 64)) and not pays(3, 30000, (2048, 5632, 16, 2, 128))
    assert not pays(8, 3000, (2560, 6912, 32, 32, 80))
    for rows in (3, 4, 8):
        assert pays(rows, 30000, (4096, 14336, 32, 8, 128)) and pays(rows, 16000, (4096, 11008, 32, 32, 128))
    assert pays(8, 30000, small, window=1024) and pays(8, 30000, small, seqs=7)
