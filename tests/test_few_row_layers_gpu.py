"""Few-row steps of plain layers launched by one native call (ops/few_row_layers.py) against the same kernels
launched one by one: the same bits."""
import pytest
import torch

import util

pytestmark = pytest.mark.gpu

# head sizes 16, 48, 128, 256; one to twenty query heads of a group; widths that are no multiple of 16
SHAPES = {"16": (64, 4, 4, 16, 176, 3), "48": (200, 10, 5, 48, 328, 2), "128": (256, 16, 1, 128, 400, 2),
          "256": (128, 2, 1, 256, 264, 2), "20 heads": (128, 20, 1, 32, 256, 1),
          "1032": (1032, 4, 4, 64, 1104, 2), "4096": (4096, 4, 1, 64, 40, 2)}


def _config(shape):
    import gpt_fast_amd as gfa
    hidden, heads, kv_heads, head_dim, inner, layers = SHAPES[shape]
    config = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": hidden,
              "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": kv_heads,
              "head_dim": head_dim, "intermediate_size": inner, "vocab_size": 320,
              "max_position_embeddings": 4096, "rope_theta": 10000.0, "rms_norm_eps": 1e-5,
              "rope_scaling": None, "tie_word_embeddings": False}
    arch = gfa.config.registry.architecture_of(config)
    return arch, arch.read_config(config)


def _engine(tmp_path, shape, dtype="bfloat16"):
    import gpt_fast_amd as gfa
    arch, config = _config(shape)
    gfa.write_random_model(str(tmp_path), arch, config, seed=5, dtype=dtype, std=0.05)
    return gfa.Engine.from_folder(str(tmp_path), dtype=dtype, device="cuda:0", max_tokens=16384)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_one_call_launches_what_the_layers_launch(tmp_path, shape, dtype, monkeypatch):
    """float32: the norms, the rotation and the gate are worked out inside the products, to the same bits."""
    _same_bits(_engine(tmp_path, shape, dtype), SHAPES[shape][5], monkeypatch)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("shape,window,rotary,activation", [("16", 3, 8, "gelu_tanh"), ("128", 70, 64, "silu"), ("48", None, 2, "gelu_tanh"),
                                                            ("1032", 1, 30, "gelu_tanh"), ("4096", 100, 64, "gelu_tanh")])
def test_with_a_window_a_part_of_the_rotation_and_the_other_gate(shape, window, rotary, activation, dtype, monkeypatch):
    import dataclasses
    import gpt_fast_amd as gfa
    from gpt_fast_amd.weights.random_init import random_parameters
    arch, config = _config(shape)
    plan = arch.plan(config)

    def changed(layer):
        position = dataclasses.replace(layer.mixer.position, rotary_dim=rotary)
        return dataclasses.replace(layer, mixer=dataclasses.replace(layer.mixer, window=window, position=position),
                                   feed_forward=dataclasses.replace(layer.feed_forward, activation=activation))
    plan = dataclasses.replace(plan, layers=[changed(layer) for layer in plan.layers])
    params = random_parameters(arch.bindings(config), 5, dtype, "cuda:0", std=0.05, norm_std=0.1, tie=False)
    _same_bits(gfa.Engine.from_plan(plan, params, dtype, "cuda:0", max_tokens=16384), SHAPES[shape][5], monkeypatch)


def _same_bits(engine, n_layers, monkeypatch):
    import gpt_fast_amd as gfa
    from gpt_fast_amd.ops import few_row_layers as F
    calls, run = [], F.run_layers
    monkeypatch.setattr(F, "run_layers", lambda layers, *a, **k: (calls.append(len(layers)), run(layers, *a, **k))[1])
    ends = list(engine.model.few_rows.ends)
    assert ends == [n_layers] * n_layers
    # held tokens, then the tokens of the step: one each (a context that is split among them), a short prompt, both
    # together, a prompt whose attention is the tiled kernel's; in float32 the products make the norms themselves for some
    # of these and not for others
    steps = [([2100], [1]), ([31, 64, 5], [1, 1, 1]), ([3] * 16, [1] * 16), ([0], [5]), ([40, 0], [1, 9]), ([0], [16])]
    for held, new in steps:
        got = []
        for apart in (False, True):
            engine.model.few_rows.ends = [0] * len(ends) if apart else ends
            slots = [engine.start_sequence() for _ in held]
            before = [gfa.Entry(s, util.random_tokens(320, n, 7 + n)) for s, n in zip(slots, held) if n]
            if before:
                engine.step(before)
            del calls[:]
            got.append(engine.step([gfa.Entry(s, util.random_tokens(320, n, 50 + i), want=list(range(n)))
                                    for i, (s, n) in enumerate(zip(slots, new))]))
            assert calls == ([] if apart else [n_layers])
            for s in slots:
                engine.end_sequence(s)
        assert torch.isfinite(got[0]).all()
        assert torch.equal(got[0], got[1]), (held, new)


def test_seventeen_rows_and_tapped_steps_go_the_general_way(tmp_path, monkeypatch):
    import gpt_fast_amd as gfa
    from gpt_fast_amd.ops import few_row_layers as F
    engine = _engine(tmp_path, "16")
    monkeypatch.setattr(F, "run_layers", lambda *a, **k: pytest.fail("not for this step"))
    slot = engine.start_sequence()
    engine.step([gfa.Entry(slot, util.random_tokens(320, 17, 1), want=[16])])
    seen = []
    engine.model.tap = lambda n, rows: seen.append(n)
    engine.step([gfa.Entry(slot, [3], want=[0])])
    assert seen == [0, 1, 2]
