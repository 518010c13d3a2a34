"""Layers launched from the list of a layer like them against the same layers run one by one, without a GPU: real models, plans
and wrappers over entry points that compute nothing.  What a call would write is taken to be a name made of the entry point, its
numbers and what it reads, so that two ways of launching a step agree on the names in the logits and in the caches exactly
where every kernel reads the same things in the same width."""

import functools
import glob
import hashlib
import os
import re

import pytest
import torch

from atomserve_amd.cache.manager import CacheManager
from atomserve_amd.config.registry import architecture_for
from atomserve_amd.engine.batch import Row
from atomserve_amd.engine.runner import ModelRunner
from atomserve_amd.kernels import build, lib, ops
from atomserve_amd.models.decoder import DecoderModel
from atomserve_amd.weights import random_checkpoint
from atomserve_amd.weights.loader import DictSource, bind_checkpoint


def _signatures() -> dict:
    """entry point -> per argument (its name, None for a number, else whether it is only read)."""
    found = {}
    for path in glob.glob(os.path.join(build.CSRC, "*.hip")):
        with open(path) as f:
            for name, args in re.findall(r'extern "C" int (as_\w+)\(([^)]*)\)', f.read()):
                found[name] = [(a.split()[-1].lstrip("*"), ("const" in a) if "*" in a else None) for a in args.split(",") if a.strip()]
    return found


SIGNATURES = _signatures()
# what a kernel changes in place, by the argument's name; an `out` is written whole unless a second kernel fills its other rows
IN_PLACE = {"x", "state", "history", "k_pages", "v_pages"}
IN_PLACE_OF = {"as_delta_prepare": {"qkv"}, "as_delta_chunks": {"out"}}


class Names:
    """Stands for the GPU: what lies at which address, as names."""

    def __init__(self):
        self.at, self.calls = {}, 0

    def call(self, entry, *args):
        if entry == "as_blas_plan":
            return 1
        read, written, numbers = [], [], []
        self.calls += 1
        for i, ((name, const), value) in enumerate(zip(SIGNATURES[entry], args, strict=True)):
            if const is None:
                numbers.append((name, value))
            elif name in ("stream", "workspace"):
                pass
            elif not value:
                read.append((name, None))
            else:
                if const or name in IN_PLACE or name in IN_PLACE_OF.get(entry, ()):
                    read.append((name, self.at.get(value, "?")))
                if not const:
                    written.append((name, value))
        made = hashlib.sha256(repr((entry, numbers, read)).encode()).hexdigest()
        for name, address in written:
            self.at[address] = (made, name)
        return 0


@pytest.fixture
def gpu(monkeypatch):
    """A GPU of names: `ops` takes tensors in host memory for its own, and no two tensors of a step share an address."""
    names, kept, real = Names(), [], torch.empty

    def check(t, name, dtype=None, shape=None):
        assert isinstance(t, torch.Tensor) and t.is_contiguous(), name
        assert dtype is None or t.dtype is dtype or (isinstance(dtype, tuple) and t.dtype in dtype), name
        assert shape is None or (len(shape) == t.dim() and all(s in (None, d) for s, d in zip(shape, t.shape))), name

    def empty(*args, **how):
        kept.append(real(*args, **how))
        return kept[-1]

    entry = lambda name: functools.partial(names.call, name)  # noqa: E731
    monkeypatch.setattr(lib, "entry", entry)
    monkeypatch.setattr(ops, "entry", entry)
    monkeypatch.setattr(ops, "_check", check)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_compute_units", 256)
    monkeypatch.setattr(ops, "_library_workspace", lambda device: kept[0])
    monkeypatch.setattr(ops.Streamed, "possible", staticmethod(lambda w: w.dtype == torch.bfloat16 and w.shape[0] % 16 == 0 and w.shape[1] % 64 == 0))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch, "empty", empty)
    torch.empty(1)
    return names


def steps(gpu, raw, weights, dtype, listed, change=None):
    """What a prompt, a portion beside it and short rows leave in the logits, the pages and the states, and the number of calls."""
    arch = architecture_for(raw)
    config = arch.parse_config(raw)
    model = DecoderModel(arch.build_plan(config), dtype, "cpu")
    bind_checkpoint(model, arch, config, DictSource(weights))
    model.env.products.fix()
    if change is not None:
        change(model)
    if not listed:
        model.stretches = None
    runner = ModelRunner(model, CacheManager(model.cache_requests(), 16, 64, 8))
    gpu.at.clear()
    for i, block in enumerate(model.blocks):
        for part, p in block.parts().items():
            for attr, v in vars(p).items():
                for kind, t in (("rows", v),) if isinstance(v, torch.Tensor) else (("rows", v.rows), ("wave", v.wave)) if isinstance(v, ops.Streamed) else ():
                    if t is not None:
                        gpu.at.setdefault(t.data_ptr(), ("weight", i, part, attr.removesuffix("_weight"), kind, t.dtype))
    cached = []
    for ident, (kind, _, _) in runner.manager.group_of_cache.items():
        for t in runner.pools.pages(ident)[1:] if kind == "paged" else runner.pools.state_of(ident)[1:]:
            cached.append(t.data_ptr())
            gpu.at[cached[-1]] = ("cache", ident, len(cached))
    held, out, calls, kept = {}, [], [], set(gpu.at)
    for step in ([("a", 40)], [("a", 1), ("b", 90)], [("a", 3), ("c", 5)]):
        rows = []
        for rid, n in step:
            cache, at = held.get(rid) or (runner.manager.new_request(), 0)
            assert runner.manager.reserve(cache, at, n)
            rows.append(Row(list(range(n)), at, cache.tables, [n - 1], cache.state_slot))
            held[rid] = (cache, at + n)
        gpu.at = {address: name for address, name in gpu.at.items() if address in kept}  # of the step before nothing else is left
        before = gpu.calls
        out.append(gpu.at[runner.step(rows).data_ptr()])
        calls.append(gpu.calls - before)
    return out, [gpu.at[address] for address in cached], calls


def qwen3(layers):
    return {"architectures": ["Qwen3ForCausalLM"], "vocab_size": 300, "hidden_size": 128, "intermediate_size": 256,
            "num_hidden_layers": layers, "num_attention_heads": 4, "num_key_value_heads": 2, "head_dim": 64, "rms_norm_eps": 1e-6,
            "rope_theta": 1e4, "tie_word_embeddings": False, "max_position_embeddings": 4096}  # fmt: skip


def table_experts(layers, times):
    delta = {"heads": 2, "kv_heads": 1, "dim": 64, "vdim": 64, "conv": 3}
    moe = {"kind": "moe", "expert": {"ff": 64}, "router": {"experts": 4, "top": 2}}
    raw = {"architecture": "Dozusun", "vocab": 300, "width": 128, "norm": {"eps": 1e-6},
           "layers": [{"type": "delta", "mixer": delta, "mlp": moe}] * layers}  # fmt: skip
    return raw if times == 1 else dict(raw, loop={"start": 0, "stop": layers, "times": times})


def checkpoint(raw, dtype):
    arch = architecture_for(raw)
    return random_checkpoint(arch, arch.parse_config(raw), seed=3, dtype=dtype, device="cpu", std=0.05)


@pytest.mark.parametrize("layers,times", [(4, 1), (2, 2), (3, 2), (2, 3), (3, 3), (5, 2)])
def test_looped_layers_choose_experts_by_their_own_tables(gpu, layers, times):
    """A layer that comes round again after its stretch has been repeated finds no other layer's routes under its table."""
    raw = table_experts(layers, times)
    weights = checkpoint(raw, torch.float32)
    assert steps(gpu, raw, weights, torch.float32, True)[:2] == steps(gpu, raw, weights, torch.float32, False)[:2]


QK, NORMS = ("self_attn.q_norm", "self_attn.k_norm"), ("input_layernorm", "post_attention_layernorm")
WIDER = {"two layers' norms": (NORMS, (3, 4)), "the last layer's norms": (NORMS, (5,)), "one layer's q and k gains": (QK, (2,)),
         "all q and k gains but one layer's": (QK, (0, 1, 3, 4, 5)), "every second layer's gains": (QK + NORMS, (0, 2, 4)),
         "the first layer's gains": (QK + NORMS, (0,)), "the written-down layer's gains": (QK + NORMS, (1,))}  # fmt: skip


@pytest.mark.parametrize("which", sorted(WIDER))
def test_gains_are_read_in_the_width_they_are_stored_in(gpu, which):
    """A 16-bit model whose checkpoint keeps the gains of some layers in 32 bits: every layer's are read in their own width."""
    raw = qwen3(6)
    weights = checkpoint(raw, torch.bfloat16)
    names, layers = WIDER[which]
    for i in layers:
        for name in names:
            weights[f"model.layers.{i}.{name}.weight"] = weights[f"model.layers.{i}.{name}.weight"].float()
    assert steps(gpu, raw, weights, torch.bfloat16, True) == steps(gpu, raw, weights, torch.bfloat16, False)


def _without_copy(model):
    model.blocks[3].ffn.down.wave = None


def _plain_matrix(model):
    model.blocks[4].mixer.o = model.blocks[4].mixer.o_weight


def _wider_gain(model):
    model.blocks[5].ffn_norm.weight = model.blocks[5].ffn_norm.weight.float()


def _another_shape(model):  # what the wrappers refuse for the layer alone
    model.blocks[4].mixer_norm.weight = torch.ones(64, dtype=torch.bfloat16)


def _another_layout(model):
    model.blocks[4].mixer_norm.weight = torch.ones(256, dtype=torch.bfloat16)[::2]


@pytest.mark.parametrize("change", [_without_copy, _plain_matrix, _wider_gain])
def test_layers_that_were_changed_run_themselves(gpu, change):
    """A matrix without its copy, a plain tensor in a matrix's place, a gain of another width: what a layer alone would launch."""
    raw = qwen3(6)
    weights = checkpoint(raw, torch.bfloat16)
    assert steps(gpu, raw, weights, torch.bfloat16, True, change) == steps(gpu, raw, weights, torch.bfloat16, False, change)


@pytest.mark.parametrize("change", [_another_shape, _another_layout])
@pytest.mark.parametrize("listed", [True, False])
def test_what_the_wrappers_refuse_stays_refused(gpu, change, listed):
    raw = qwen3(6)
    with pytest.raises(AssertionError, match="weight"):
        steps(gpu, raw, checkpoint(raw, torch.bfloat16), torch.bfloat16, listed, change)


def test_a_list_is_made_again_only_for_what_it_fits(gpu):
    """Layers of equal sizes are launched from the list: as many calls, and the wrappers' checks run for the first layers alone."""
    raw, checked = qwen3(6), []
    weights = checkpoint(raw, torch.bfloat16)
    real = ops._check
    ops._check = lambda t, name, dtype=None, shape=None: (checked.append(name), real(t, name, dtype, shape))
    try:
        listed = steps(gpu, raw, weights, torch.bfloat16, True)
        few = len(checked)
        alone = steps(gpu, raw, weights, torch.bfloat16, False)
    finally:
        ops._check = real
    assert listed == alone and few < 0.7 * (len(checked) - few)


def test_a_list_of_calls_is_made_again_as_it_was_written_down():
    """Entry points with few and many integers, floats anywhere among them and none: every argument arrives, the patched ones
    as the targets say, and a status that is not zero ends the list and names its call."""
    from ctypes import CFUNCTYPE, c_float, c_int, c_longlong, c_size_t, c_void_p

    from atomserve_amd.kernels.lib import KernelError, Launches

    shapes = [(c_void_p,), (c_float,), (), (c_int, c_float, c_void_p, c_float, c_longlong, c_void_p, c_int, c_int, c_size_t, c_float, c_void_p),
              (c_void_p, c_int) * 15, (c_int,) * 5 + (c_float,) + (c_void_p,) * 20 + (c_float, c_int)]  # fmt: skip
    seen, status, made, kept = [], [0], Launches(), []
    made.calls = []
    for i, kinds in enumerate(shapes):
        def entry(*got, i=i):
            seen.append((i, [0 if v is None else v for v in got]))
            return status[0] if i == 4 else 0

        kept.append(CFUNCTYPE(c_int, *kinds)(entry))
        args = [0.5 + n if kind is c_float else None if kind is c_void_p and n % 3 == 2 else (1 << 40) + 8 * n if kind is c_void_p else -3 - n
                if kind is not c_size_t else 7 for n, kind in enumerate(kinds)]  # fmt: skip
        made.calls.append((f"call {i}", kept[-1], args))
    sources = [(1 << 40) + 8 * n for n in (0, 4, 6, 6)]
    made.aim(sources)
    assert made.met == [0, 1, 2, 3] and made.fits([1, 2, 3, 3]) and not made.fits([1, 2, 3, 4])
    targets = [11, 22 << 40, 33, 33]
    made.again(targets)
    at = dict(zip(sources, targets))
    assert seen == [(i, [0 if v is None else at.get(v, v) for v in args]) for i, (_, _, args) in enumerate(made.calls)]
    seen.clear()
    status[0] = -2
    with pytest.raises(KernelError, match="call 4"):
        made.again(targets)
    assert [i for i, _ in seen] == [0, 1, 2, 3, 4]
    made.program[1] = 99  # a call of more integers than the list allows
    seen.clear()
    with pytest.raises(KernelError, match="as_launch_list"):
        made.again(targets)
    assert not seen


@pytest.mark.parametrize("kinds", [("i",) * 33, ("f",) * 5, ("i", "d", "i"), ("p", "f", "d"), ("i",) * 32 + ("f",) * 4])
def test_calls_that_no_list_holds_are_made_one_by_one(kinds):
    """More integers or floats than a call of a list has, or floats of 64 bits: every argument arrives all the same, the patched ones as the
    targets say, and a status that is not zero names its call.  (The last one is as large as a list's calls come.)"""
    from ctypes import CFUNCTYPE, c_double, c_float, c_int, c_void_p

    from atomserve_amd.kernels.lib import KernelError, Launches

    types = [{"i": c_int, "f": c_float, "d": c_double, "p": c_void_p}[k] for k in kinds]
    seen, status, made = [], [0], Launches()

    def entry(*got):
        seen.append(list(got))
        return status[0]

    function = CFUNCTYPE(c_int, *types)(entry)
    function.argtypes = types  # a list, as the entry points' are
    args = [0.5 + n if k in "fd" else 1000 + n for n, k in enumerate(kinds)]
    if "d" in kinds:
        args[kinds.index("d")] = 1.0 + 2.0**-40
    made.calls = [("the call", function, args)]
    sources = [args[n] for n, k in enumerate(kinds) if k in "ip"][-1:]
    made.aim(sources)
    made.again([7] * len(sources))
    assert seen == [[7 if v in sources else v for v in args]]
    status[0] = -2
    with pytest.raises(KernelError, match="the call"):
        made.again([7] * len(sources))
    assert (made.program is None) == (len(kinds) != 36)
    seen.clear()
    status[0] = 0
    args[-1] = types[-1](3)  # no plain number
    made.calls = [("the call", function, args)]
    made.aim([])
    made.again([])
    assert made.program is None and seen == [[*args[:-1], 3]]
