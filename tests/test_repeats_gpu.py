"""Layers launched from the list of a layer like them against the same layers run one by one: the same bits in the logits, the
pages and the states, whatever the step brings."""

import pytest
import torch

from atomserve_amd.cache.manager import CacheManager
from atomserve_amd.config.registry import architecture_for
from atomserve_amd.engine.batch import Row
from atomserve_amd.engine.runner import ModelRunner
from atomserve_amd.models.decoder import DecoderModel
from atomserve_amd.weights import random_checkpoint
from atomserve_amd.weights.loader import DictSource, bind_checkpoint

pytestmark = pytest.mark.gpu


def qwen3(layers, hidden=256):
    return {"architectures": ["Qwen3ForCausalLM"], "vocab_size": 300, "hidden_size": hidden, "intermediate_size": 2 * hidden,
            "num_hidden_layers": layers, "num_attention_heads": 4, "num_key_value_heads": 2, "head_dim": 64, "rms_norm_eps": 1e-6,
            "rope_theta": 1e4, "tie_word_embeddings": False, "max_position_embeddings": 4096}  # fmt: skip


def dozusun(kinds):
    side = {"left": {"heads": 2, "kv_heads": 1, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": 40}}, "left_scale": 0.8,
            "right_scale": 0.9, "right": {"width": 128, "blocks": 2, "conv": 4}}  # fmt: skip
    delta = {"heads": 2, "kv_heads": 1, "dim": 64, "vdim": 64, "conv": 3}
    moe = {"kind": "moe", "expert": {"ff": 64}, "router": {"experts": 4, "top": 2}}
    layers = {"p": {"type": "parallel", "mixer": side, "mlp": {"kind": "dense", "ff": 128}},
              "d": {"type": "delta", "mixer": delta, "mlp": moe}, "n": {"type": "delta", "mixer": delta}}  # fmt: skip
    return {"architecture": "Dozusun", "vocab": 300, "width": 128, "norm": {"eps": 1e-6}, "layers": [layers[k] for k in kinds]}


CASES = {"qwen3-6": (qwen3(6), (1, 1, 3)), "qwen3-3": (qwen3(3), None), "qwen3-5": (qwen3(5, 512), (1, 1, 2)),
         "dozusun-pairs": (dozusun("pdpdpdpd"), (1, 2, 2)), "dozusun-alone": (dozusun("nnnn"), (1, 1, 2)),
         "dozusun-mixed": (dozusun("pddnpd"), (1, 1, 1)),
         "dozusun-looped": (dict(dozusun("ddd"), loop={"start": 0, "stop": 3, "times": 2}), (1, 1, 2)),
         "dozusun-looped-twice": (dict(dozusun("ddd"), loop={"start": 0, "stop": 3, "times": 3}), (1, 2, 2))}  # fmt: skip


# whose gains are stored in the other width: (names, layers)
WIDER = {"two layers' norms": (("input_layernorm", "post_attention_layernorm"), (3, 4)), "one layer's q and k gains": (("self_attn.q_norm", "self_attn.k_norm"), (2,)),
         "all q and k gains but one layer's": (("self_attn.q_norm", "self_attn.k_norm"), (0, 1, 3, 4, 5))}  # fmt: skip


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", sorted(CASES))
def test_layers_from_a_list_are_the_layers(name, dtype):
    check_layers(*CASES[name], dtype)


@pytest.mark.parametrize("which", sorted(WIDER))
def test_layers_with_gains_of_other_widths_are_the_layers(which):
    def change(weights):
        names, layers = WIDER[which]
        for name in [f"model.layers.{i}.{n}.weight" for i in layers for n in names]:
            weights[name] = weights[name].float()

    check_layers(*CASES["qwen3-6"], torch.bfloat16, change)


def check_layers(raw, covered, dtype, change=None):
    arch = architecture_for(raw)
    config = arch.parse_config(raw)
    weights = random_checkpoint(arch, config, seed=3, dtype=dtype, device="cuda:0", std=0.05)
    if change is not None:
        change(weights)

    def steps(listed: bool):
        model = DecoderModel(arch.build_plan(config), dtype, "cuda:0")
        bind_checkpoint(model, arch, config, DictSource(weights))
        model.env.products.fix()
        assert model.stretches == covered
        if not listed:
            model.stretches = None
        manager = CacheManager(model.cache_requests(), 16, 64, 8)
        runner = ModelRunner(model, manager)
        gen, held, out = torch.Generator().manual_seed(1), {}, []
        # (request, tokens): few rows, prompts around the products' and the chunks' borders, portions beside decoding requests
        for step in ([("a", 5)], [("b", 14)], [("c", 17)], [("a", 1), ("d", 40)], [("b", 100), ("c", 1), ("a", 3)], [("e", 200)],
                     [("a", 1), ("b", 1), ("c", 30), ("e", 90)], [("a", 1), ("b", 1), ("e", 1)], [("d", 9), ("a", 2)]):  # fmt: skip
            rows = []
            for rid, n in step:
                cache, at = held.get(rid) or (manager.new_request(), 0)
                assert manager.reserve(cache, at, n)
                tokens = torch.randint(300, (n,), generator=gen).tolist()
                rows.append(Row(tokens, at, cache.tables, [0, n - 1][: min(n, 2)], cache.state_slot))
                held[rid] = (cache, at + n)
            out.append(runner.step(rows).clone())
        return out, runner.pools.paged, [t[:, :-1] for t in runner.pools.state]

    (a, pages_a, states_a), (b, pages_b, states_b) = steps(True), steps(False)
    for i, (x, y) in enumerate(zip(a, b)):
        assert torch.equal(x, y), f"step {i}"
    assert all(torch.equal(x, y) for x, y in zip(pages_a + states_a, pages_b + states_b))


def test_a_layer_that_is_watched_runs_itself():
    raw, _ = CASES["qwen3-6"]
    arch = architecture_for(raw)
    config = arch.parse_config(raw)
    model = DecoderModel(arch.build_plan(config), torch.float32, "cuda:0")
    bind_checkpoint(model, arch, config, DictSource(random_checkpoint(arch, config, seed=3, dtype=torch.float32, device="cuda:0")))
    manager = CacheManager(model.cache_requests(), 16, 8, 1)
    runner = ModelRunner(model, manager)
    cache = manager.new_request()
    manager.reserve(cache, 0, 20)
    rows = [Row(list(range(20)), 0, cache.tables, [19])]
    want, seen = runner.step(rows).clone(), []
    for i in (1, 3):
        inner = model.blocks[i].forward
        model.blocks[i].forward = lambda *a, inner=inner, i=i, **k: (seen.append(i), inner(*a, **k))[1]
    assert torch.equal(runner.step(rows), want) and seen == [1, 3]
