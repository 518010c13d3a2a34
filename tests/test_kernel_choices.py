"""Which kernel, and cut how, for which sizes: the decisions of `kernels/ops.py` that need no GPU.  They
decide speed only (every route gives the same result within rounding, which the GPU tests hold them to); the
vectors here pin what the sizes say on an MI355X's 256 compute units, so that a change of a limit or a cost
shows as a change of a choice."""

import pytest
import torch

from atomserve_amd.kernels import ops

BF16, F32 = torch.bfloat16, torch.float32


@pytest.fixture(autouse=True)
def on_256_compute_units(monkeypatch):
    monkeypatch.setattr(ops, "_compute_units", 256)
    ops._prefill_plan_of.cache_clear()


def test_how_a_prompt_steps_attention_is_cut():
    """A portion behind a long prefix is few long items: cut along the keys, into the more pieces the fewer the
    items, a wave owning 32 queries where that still fills the GPU and 16 where only that does.  A lone prompt, a
    short context, a window that keeps every item short: not cut."""
    plan = lambda tokens, H, context, **kw: ops._prefill_plan(-(-tokens // 64), H, 8, 128, context, **kw)
    assert plan(512, 32, 16384) == (2, 4, 64)  # 128 items of 256 rounds: four pieces of 64 fill the 512 places
    assert plan(1024, 32, 16384) == (2, 2, 128)
    assert plan(512, 16, 16384) == (2, 8, 32)  # half the heads: twice the pieces
    assert plan(64, 32, 20000) == (1, 8, 40)  # one tile: 16 queries to a wave make twice the workgroups
    assert plan(512, 32, 4096) == (1, 2, 32)
    for tokens in (256, 512, 1024, 2048, 4096, 8192, 16384):  # lone prompts: whole
        assert plan(tokens, 32, tokens)[1:] == (1, 0) and plan(tokens, 16, tokens)[1:] == (1, 0)
    assert plan(1024, 32, 1024)[0] == 1 and plan(8192, 32, 8192)[0] == 2
    assert plan(512, 32, 1024)[1:] == (1, 0)  # 16 rounds: too short to pay for the merge
    assert plan(512, 32, 8192, window=512)[1:] == (1, 0)
    # as many items as places: whole if all are as long as the longest, cut if most are short
    assert plan(2048, 32, 16384, tile_keys=32 * 16384)[1] == 1 and plan(2048, 32, 16384, tile_keys=32 * 4000)[1] > 1
    # whatever is chosen, the pieces cover the longest item and have at least the rounds the kernel asks for
    for tokens, H, context in ((64, 8, 700), (512, 64, 40000), (130, 40, 9000), (4096, 16, 4096), (64, 32, 128)):
        for forced in (None, 2, 3, 5, 8):
            ops.PREFILL_PIECES = forced
            try:
                kind, pieces, piece_rounds = plan(tokens, H, context)
            finally:
                ops.PREFILL_PIECES = None
            rounds = -(-context // 64)
            assert kind in (1, 2) and 1 <= pieces <= 8
            assert (pieces, piece_rounds) == (1, 0) or (piece_rounds >= 2 and pieces * piece_rounds >= rounds)


def test_how_single_queries_contexts_are_partitioned():
    """Few requests: partitions of a size by which the GPU's places are filled and the merge stays small; from
    one and a half (token, kv head) pairs per compute unit on, whole contexts."""
    assert ops.attn_fill_groups() == 384
    best = lambda groups, span: min(ops.MFMA_PARTITIONS, key=lambda part: ops._partition_cost(groups, span, part))
    assert [best(8, 2048), best(64, 2048), best(64, 500)] == [256, 256, 128]
    assert [best(8, 16384), best(64, 16384), best(8, 33000)] == [512, 2048, 1024]
    # through `_partitions`, on the CPU: sizes and buffers
    size, P, m, l, acc = ops._partitions(8, 32, 8, 128, 2048, 0, True, None, "cpu")
    assert (size, P) == (256, 8) and m.shape == (8, 32, 8) and acc.shape == (8, 32, 8, 128)
    size, P, m, l, acc = ops._partitions(64, 32, 8, 128, 2100, 0, True, None, "cpu")
    assert (size, P, m) == (2112, 1, None)  # 512 pairs: the whole context, rounded up to steps of 32 keys
    size, P, *_ = ops._partitions(8, 32, 8, 128, 5000, 1024, True, None, "cpu")
    assert size == 256 and P == 5  # a window: the keys it shows (in whole steps of 32) decide the size and how many there are
    size, P, *_ = ops._partitions(8, 32, 8, 128, 5000, 1024, True, 128, "cpu", keep_first=100)
    assert size == 128 and P == 10  # and the kept first ones
    assert ops._seen_keys(5000, 1, 0, True) == 32 and ops._seen_keys(5000, 2, 5, True) == 96 and ops._seen_keys(5000, 2, 5, False) == 7
    assert ops._seen_keys(90, 100, 30, True) == 96 and ops._seen_keys(90, 0, 0, True) == 90
    with pytest.raises(ops.KernelError, match="multiples of 32"):
        ops._partitions(8, 32, 8, 128, 2048, 0, True, 100, "cpu")


def test_short_contexts_are_walked_whole():
    """Up to 256 keys a workgroup of a (token, kv head) pair is faster than partitions and their merge, whoever asks; the captured
    step of few rows has a form for them."""
    from atomserve_amd.engine.runner import DecodeGraphs

    for rows in (1, 8, 32):
        assert ops._partitions(rows, 16, 8, 128, 256, 0, True, None, "cpu")[1] == 1
        assert ops._partitions(rows, 16, 8, 128, 512, 0, True, None, "cpu")[1] > 1
    bounds = lambda n, context: DecodeGraphs._bounds(DecodeGraphs, n, context)  # noqa: E731
    assert bounds(1, 1024) == bounds(32, 1024) == (256, 1024) and bounds(48, 1024) == (1024,) and bounds(1, 2048) == (2048,)


def test_forms_of_a_captured_bucket():
    """A bucket is captured in two forms only where the attention of some layer cuts its longer contexts and not the short ones."""
    from types import SimpleNamespace

    from atomserve_amd.engine.runner import DecodeGraphs
    from atomserve_amd.models.decoder import DecoderModel
    from atomserve_amd.parts.attention import Attention
    from atomserve_amd.parts.base import Mixer

    def graphs(*heads, dtype=BF16):
        mixer = SimpleNamespace(single_queries=lambda: heads)
        model = SimpleNamespace(env=SimpleNamespace(dtype=dtype), blocks=[SimpleNamespace(parts=lambda: {"mixer": mixer})])
        model.contexts_cut = lambda *how: DecoderModel.contexts_cut(model, *how)
        made = DecodeGraphs.__new__(DecodeGraphs)
        made.runner, made.two_forms = SimpleNamespace(model=model, manager=SimpleNamespace(block_size=16)), {}
        return made

    two, one = (256, 1024), (1024,)
    g = graphs((16, 8, 128, 0, 0))
    assert [g._forms(n, 1024) for n in (1, 32, 48)] == [two, two, one] and g._forms(1, 2048) == (2048,) and g.two_forms == {1: True, 32: True}
    assert graphs()._forms(1, 1024) == one  # no paged attention of this kind
    assert [graphs((32, 16, 128, 0, 0))._forms(n, 1024) for n in (16, 32)] == [two, one]  # 32 x 16 workgroups fill the GPU
    assert graphs((16, 8, 128, 200, 0))._forms(1, 1024) == one  # a window that both contexts fill
    assert graphs((16, 8, 128, 0, 0), (16, 8, 128, 200, 0), dtype=F32)._forms(4, 1024) == two
    spec = SimpleNamespace(num_heads=16, num_kv_heads=8, head_dim=128, window=64)
    assert Attention.single_queries(SimpleNamespace(spec=spec)) == ((16, 8, 128, 64, 0),) and Mixer.single_queries(None) == ()


def test_how_products_of_17_to_128_rows_are_tiled():
    """Tiles of 64 weight rows, K cut into as many ranges of whole chunks as fill the compute units; the gated
    product's tile width by what the longest path loads."""
    assert ops.gemm_split_plan(64, 4096, 4096, BF16) == (4, 4)
    assert ops.gemm_split_plan(64, 4096, 12288, BF16) == (4, 4)
    assert ops.gemm_split_plan(32, 1024, 3072, BF16) == (4, 12)
    assert ops.gemm_split_plan(128, 5120, 25600, BF16) == (4, 3)
    assert ops.gemm_split_plan(8, 4096, 4096, BF16) is None  # few rows: the few-rows kernels'
    assert ops.gemm_split_plan(64, 4096, 4000, BF16) is None  # K in chunks of 256
    assert ops.gemm_split_plan(64, 4096, 4096, F32) is None
    assert [ops._gated_tile_strips(*case) for case in ((64, 12288), (64, 3072), (128, 25600))] == [6, 2, 8]


def test_tiles_of_experts_pairs():
    """Tiles of 128 pairs belong to the kernel that streams weights alone, both products of a layer on it, and there to enough pairs."""
    weights = lambda rows, k, experts=16, dtype=ops.BF16: torch.empty(experts, rows, k, dtype=dtype, device="meta")  # noqa: E731

    class At:  # weights that start where they are told to
        def __init__(self, w, at):
            self.shape, self.dtype, self.at, self.numel = w.shape, w.dtype, at, w.numel

        def data_ptr(self):
            return self.at

    def tile(pairs, first, second, gated=True, at=(0, 0)):
        return ops.moe_tile(pairs, At(first, at[0]), At(second, at[1]), gated)

    first, second = weights(3072, 2048), weights(2048, 1536)
    assert [tile(16 * n, first, second) for n in (1, 31, 32, 300)] == [64, 64, 128, 128]
    small = weights(1536, 1024), weights(1024, 768)
    assert [tile(16 * n, *small) for n in (1, 31, 32, 300)] == [64, 64, 128, 128]
    assert tile(16 * 300, weights(3072, 2048, dtype=ops.F32), weights(2048, 1536, dtype=ops.F32)) == 64
    for rows, k, out in ((5760, 2880, 2880), (2000, 1024, 1024), (2048, 1000, 1024), (2048, 1024, 1000), (3080, 2048, 2048)):
        assert tile(16 * 300, weights(rows, k), weights(out, rows // 2)) == 64
    assert tile(16 * 300, first, second, at=(8, 0)) == tile(16 * 300, first, second, at=(0, 8)) == 64
    assert tile(16 * 300, weights(4096, 4096), weights(4096, 4096), gated=False) == 128
    assert tile(300, weights(1 << 18, 8192, 1), weights(8192, 1 << 17, 1)) == 64  # an expert beyond 32-bit offsets


@pytest.mark.parametrize("first,second", [(3072, 4096), (8192, 2048)])  # the wider input: gate and up's, down's
def test_pairs_whose_rows_pass_4_gib_are_not_in_tiles_of_128(first, second):
    """The kernel of large tiles finds its pairs' rows at 32-bit offsets and takes tiles of 128 up to 0xf0000000 bytes of them; beyond, such a route
    would go to the kernel for all sizes, which is slower than tiles of 64."""

    class Weights:
        def __init__(self, *shape):
            self.shape, self.dtype, self.numel, self.data_ptr = shape, BF16, lambda: shape[0] * shape[1] * shape[2], lambda: 0

    inner = first // 2
    up, down = Weights(64, first, second), Weights(64, second, inner)
    widest = max(second, inner)
    most = 0xF0000000 // (2 * widest) // 128 - 64  # tiles of pairs: one more for every expert is counted
    assert ops.moe_tile(128 * most, up, down, True) == 128 and ops.moe_tile(128 * most + 1, up, down, True) == 64


def test_which_plain_products_take_the_tile_kernel_without_trials(monkeypatch):
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    strips = ops._plain_tile_strips
    for rows in (17, 48, 64):
        assert [strips(rows, n, k, ops.BF16) for n, k in ((4096, 1024), (6144, 4096), (8192, 5120), (8208, 5120), (10240, 5120))] == [2, 2, 2, 4, 4]
        assert [strips(rows, n, k, ops.BF16) for n, k in ((4080, 1024), (4096, 8192), (2560, 9728))] == [0, 0, 0]
        assert strips(rows, 6144, 4096, ops.F32) == 0
    assert strips(16, 6144, 4096, ops.BF16) == strips(65, 6144, 4096, ops.BF16) == 0


def test_plain_products_that_trials_decide(monkeypatch):
    """Where the library wins at some of 17 to 64 rows: few outputs of a longer K, and more outputs than one round of workgroups holds."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    for rows in (17, 32, 64):
        for n, k in ((4096, 2560), (4096, 4096), (5104, 4096), (16400, 1024), (24576, 2048), (32768, 4096)):
            assert ops._plain_tile_strips(rows, n, k, ops.BF16) == 0
        assert [ops._plain_tile_strips(rows, n, k, ops.BF16) for n, k in ((4096, 2048), (5120, 4096), (16384, 5120))] == [2, 2, 4]


class Mark:  # an event of a timed run
    def __init__(self, ms=None):
        self.ms = ms

    def query(self):
        return True

    def elapsed_time(self, end):
        return end.ms


def test_the_shortest_run_of_a_trial_decides():
    """Of the runs with the host ahead where every candidate has one; else of all but each candidate's first."""
    runs = lambda *times: [(c, Mark(), Mark(ms)) for n in range(len(times[0])) for c, ms in enumerate(t[n] for t in times)]  # noqa: E731
    assert ops._fastest_of({"runs": runs((1.0, 5.0, 5.1, 50.0), (9.0, 6.0, 6.0, 6.0))}) == 0
    assert ops._fastest_of({"runs": runs((9.0, 6.0, 6.0, 6.0), (9.0, 7.0, 40.0, 5.0))}) == 1
    assert ops._fastest_of({"runs": runs((9.0, 3.0, 6.0, 6.0), (9.0, 40.0, 5.0, 5.5)), "ahead": 4}) == 1  # the last two runs of both
    assert ops._fastest_of({"runs": runs((9.0, 3.0, 6.0), (9.0, 4.0, 5.0))[:5], "ahead": 4}) == 0  # only one candidate ran ahead
    assert ops._fastest_of({"runs": [(3, None, None)]}) == 0 and ops._fastest_of({"runs": []}) == 0


def test_the_rest_of_a_trial_runs_on_all_weights_in_turn(monkeypatch):
    met, fills = [], []

    def run(trial, a, w, out, M, N, K):
        met.append(w)
        trial["runs"].append((trial["ids"][len(trial["runs"]) % trial["count"]], Mark(), Mark(1.0)))

    monkeypatch.setattr(ops, "_trial_run", run)
    Fill = type("Fill", (), {"zero_": lambda self: fills.append(len(met)), "__getitem__": lambda self, part: self})
    monkeypatch.setattr(ops, "_library_workspace", lambda device: Fill())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: type("S", (), {"synchronize": lambda self: None})())
    rows = torch.empty(1)
    for M, done, more in ((32, 1, 4), (32, 8, 4), (2048, 6, 2), (2048, 8, 0)):
        choices, before = ops.ProductChoices(), [(n % 2, Mark(), Mark(2.0)) for n in range(done)]
        choices.trials[(M, 64, 64, BF16)] = {"count": 2, "ids": [0, 1], "runs": before, "weights": ["a", "b", "c"], "last": (rows, "c", None)}
        met.clear(), fills.clear()
        choices.settle()
        assert met == [("a", "b", "c")[(done + n) % 3] for n in range(more)] and (M, 64, 64, BF16) in choices.chosen()
        assert fills == ([0] * more + list(range(more)) if M == 32 else [])  # the queue is filled before the first run and between the runs
    with torch.inference_mode():
        space = torch.ones(8, dtype=torch.uint8)  # what a model's pass has made, cleared by a caller outside of it
    monkeypatch.setattr(ops, "_library_workspace", lambda device: space)
    choices.trials[(32, 64, 64, BF16)] = {"count": 1, "ids": [0], "runs": [], "weights": ["a"], "last": (rows, "a", None)}
    choices.settle()
    assert int(space.sum()) == 0


def test_how_rows_of_a_state_space_are_cut_into_segments():
    """One long row fills the GPU in segments, whatever short rows stand beside it; many rows of its length stay whole."""
    choose = ops._state_space_segments
    assert choose(2048, 2048, 64) == 256  # 128 heads of 64: 8 segments of 64 workgroups
    assert choose(2041, 2048, 64) == 256 and choose(1700, 2048, 64) == 256  # beside decoding requests, behind another prompt's end
    assert choose(512, 2048, 64) == 256 and choose(511, 2048, 64) == 0 and choose(256, 2048, 64) == 0
    assert choose(2048, 2048, 8) == 64 and choose(200, 200, 1) == 64 and choose(100, 100, 1) == 0 and choose(0, 5, 1) == 0
    assert choose(8192, 8192, 4096) == 0  # a row's own workgroups fill it


def test_which_32_bit_portions_run_as_prompt_tiles():
    """A tile reads its keys once for all of its queries, a single query's keys are cut into partitions: short portions behind
    long prefixes are single queries (as tiles they took longer than on the general kernel), prompts are tiles."""
    tiles = lambda tokens, context, H=16, KV=8, D=128, window=0, short=0: ops.attn_tiles_preferred(  # noqa: E731
        tokens, short, H, KV, D, context, window)
    assert [tiles(n, 8000 + n) for n in (9, 16, 64, 128, 512)] == [False, False, True, True, True]
    assert [tiles(n, n) for n in (9, 37, 64, 333, 512)] == [False, False, False, True, True]
    assert not tiles(9, 30009) and not tiles(9, 2009) and tiles(33, 2033)
    assert [tiles(n, 8000 + n, 4, 2, 64) for n in (9, 64, 128, 512)] == [False, False, False, True]
    assert not tiles(9, 8009, window=512) and tiles(128, 8128, window=512) and tiles(520, 8000, short=8)


@pytest.mark.parametrize("tokens,start,how", [(9, 8000, "single"), (9, 0, "single"), (128, 8000, "tiles"), (333, 0, "tiles"), (5, 100, "short")])
def test_the_route_of_a_32_bit_portion(monkeypatch, tokens, start, how):
    from types import SimpleNamespace

    from atomserve_amd.parts.attention import attend

    made = []
    monkeypatch.setattr(ops, "attn_single_query", lambda q, k, v, items, *args, **kw: made.append(("single", items)))
    monkeypatch.setattr(ops, "attn_prefill_f32", lambda q, k, v, tiles, *args, **kw: made.append(("tiles", tiles)))
    pages = torch.empty(1, 8, 16, 128)
    cache = SimpleNamespace(k_pages=pages, v_pages=pages.view(1, 8, 128, 16), block_tables=None, block_size=16)
    rows = SimpleNamespace(num_short_tokens=tokens if tokens <= 8 else 0, num_long_tiles=0 if tokens <= 8 else -(-tokens // 64),
                           short_tokens="short", long_tiles="long", max_short_context=start + tokens)  # fmt: skip
    step = SimpleNamespace(decode_only=False, all_tokens="all", positions=None, tok_row=None, max_context=start + tokens, split=lambda key: rows)
    attend(torch.empty(tokens, 16, 128), None, step, cache, 1.0, 0, (8, 64))
    assert made == [{"single": ("single", "all"), "tiles": ("tiles", "long"), "short": ("single", "short")}[how]]


def test_plans_of_steps_with_portions_and_single_queries(monkeypatch):
    """Pieces and partitions cover the longest item and context, and every piece and partition is one that the kernel takes."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    ops._mixed_plan.cache_clear()
    try:
        for H, KV, D in ((32, 8, 128), (40, 8, 128), (16, 1, 64), (6, 3, 64)):
            for tokens, behind, singles, context, window in ((37, 0, 1, 1, 0), (480, 7001, 32, 2049, 0), (2000, 0, 128, 400, 0), (100, 8000, 1, 8193, 0),
                                                             (300, 5000, 64, 6000, 1024), (9, 31, 3, 40, 1)):  # fmt: skip
                tiles, most = -(-tokens // 64), behind + tokens
                keys = sum(behind + min(tokens, 64 * (i + 1)) for i in range(tiles))
                kind, pieces, piece_rounds, part = ops._mixed_plan(tiles, H, KV, D, most, keys, singles, context, window, 256)
                span = min(most, window + 64) if window else most
                assert kind in (1, 2) and part % 32 == 0 and part >= 32
                assert (pieces, piece_rounds) == (1, 0) or (pieces * piece_rounds * 64 >= span and piece_rounds >= 2)
        assert ops._mixed_plan(8, 32, 8, 128, 7481, 8 * 7257, 32, 2049, 0, 256) == (2, 4, 30, 2080)
    finally:
        ops._mixed_plan.cache_clear()


@pytest.mark.parametrize("query_tiles,pieces,want", [(None, None, (2, 4, 30)), (1, None, (1, 2, 59)), (None, 5, (2, 5, 24)), (2, 1, (2, 1, 0)), (1, 99, (1, 58, 3))])
def test_forced_cuts_of_portions_hold_beside_single_queries(monkeypatch, query_tiles, pieces, want):
    """What forces a variant and a number of pieces for a step of portions alone forces them where single queries share the launch."""
    made = []
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    monkeypatch.setattr(ops, "_check", lambda *args: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_partitions", lambda *args: (args[7], 1, None, None, None))
    monkeypatch.setattr(ops, "call", lambda name, *args: made.append(args[18:21]))
    monkeypatch.setattr(ops, "PREFILL_QUERY_TILES", query_tiles)
    monkeypatch.setattr(ops, "PREFILL_PIECES", pieces)
    ops._mixed_plan.cache_clear()
    try:
        q, pages = torch.empty(512, 32, 128, dtype=torch.bfloat16), torch.empty(1, 8, 16, 128, dtype=torch.bfloat16)
        ops.attn_mixed(q, pages, pages.view(1, 8, 128, 16), torch.empty(32, dtype=torch.int32), torch.empty(8, 4, dtype=torch.int32), None, None,
                       torch.empty(33, 468, dtype=torch.int32), q, 0.1, 0, 7481, 2049, 8 * 7257)  # fmt: skip
    finally:
        ops._mixed_plan.cache_clear()
    assert made == [want]


@pytest.mark.parametrize("tiles,H,KV,D,most,keys,singles,context,forms", [
    (10, 16, 8, 128, 5446, 51841, 1, 224, {(1, 3), (1, 6), (2, 3), (2, 6)}), (48, 16, 4, 128, 6207, 226073, 1, 83, {(2, 1), (2, 3)}),
    (5, 32, 8, 128, 6044, 29716, 7, 59, {(1, 3)}), (51, 32, 8, 64, 3253, 84853, 93, 106, {(1, 1)}), (19, 6, 3, 64, 4043, 66629, 1, 38, {(1, 4), (1, 6)}),
    (20, 40, 8, 128, 5804, 20 * 5200, 1, 635, {(2, 1)})])  # fmt: skip
def test_long_portions_beside_few_or_short_contexts_are_not_slower_than_alone(monkeypatch, tiles, H, KV, D, most, keys, singles, context, forms):
    """Steps that were 14 to 32 per cent slower in one launch than in two where they were cut into eights or halves, or (the last) where portions that
    all have a place were cut at all; forms: (query tiles, pieces) that took no more than two launches by a hundredth."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    ops._mixed_plan.cache_clear()
    try:
        assert ops._mixed_plan(tiles, H, KV, D, most, keys, singles, context, 0, 256)[:2] in forms
    finally:
        ops._mixed_plan.cache_clear()


@pytest.mark.parametrize("behind,context,H", [(7001, 2049, 32), (12000, 8192, 64), (0, 300, 16)])
def test_a_plan_for_new_lengths_costs_little_on_the_host(behind, context, H):
    """The lengths of a running server's step are new ones, so a plan is made in each before its first attention is launched: no more than 120
    Python calls for all ways to cut the step (346 and 57 to 140 us with a cost worked out from the start for each way)."""
    import sys

    calls = []
    sys.setprofile(lambda frame, event, arg: calls.append(event) if event in ("call", "c_call") else None)
    try:
        ops._mixed_plan.__wrapped__(8, H, 8, 128, behind + 480, 8 * (behind + 250), 32, context, 0, 256)
    finally:
        sys.setprofile(None)
    assert len(calls) <= 120


@pytest.mark.parametrize("dtype,D,page,sight,one", [(torch.bfloat16, 128, 16, {}, True), (torch.bfloat16, 64, 16, {}, True), (torch.bfloat16, 96, 16, {}, False),
                                                    (torch.bfloat16, 128, 32, {}, False), (torch.bfloat16, 128, 16, {"softcap": 5.0}, False)])  # fmt: skip
def test_the_route_of_a_step_with_portions_and_single_queries(monkeypatch, dtype, D, page, sight, one):
    from types import SimpleNamespace

    from atomserve_amd.parts.attention import attend

    made = []
    for name in ("attn_mixed", "attn_single_query", "attn_prefill"):
        monkeypatch.setattr(ops, name, lambda *a, name=name, **kw: made.append(name))
    pages = torch.empty(1, 8, page, D, dtype=dtype)
    cache = SimpleNamespace(k_pages=pages, v_pages=pages.view(1, 8, D, page), block_tables=None, block_size=page)
    rows = SimpleNamespace(num_short_tokens=3, num_long_tiles=2, short_tokens="short", long_tiles="long", max_short_context=90, max_tile_context=100, tile_keys=164)
    step = SimpleNamespace(decode_only=False, all_tokens="all", positions=None, tok_row=None, max_context=100, split=lambda key: rows)
    attend(torch.empty(103, 16, D, dtype=dtype), None, step, cache, 1.0, 0, (8, 64), **sight)
    assert made == (["attn_mixed"] if one else ["attn_single_query", "attn_prefill"])


def test_plans_of_wide_products(monkeypatch):
    """Products of more than 128 rows: ranges of K that are none of them empty, in one round of workgroups, and no range where
    the library's whole product takes less."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    for cached in (ops._wide_plan, ops.wide_split_plan, ops.wide_gated_form):
        cached.cache_clear()
    try:
        for rows in (129, 200, 333, 512, 1000, 2409, 65536):
            for n, k in ((16, 64), (1024, 3072), (2560, 9728), (4096, 12288), (5120, 25600), (4096, 64), (151936, 4096)):
                plan = ops.wide_split_plan(rows, n, k)
                if plan is not None:
                    tm, tn, each, *_ = ops.WIDE_FORMS[plan[0]]
                    units = -(-(k // 64) // plan[1])
                    assert plan[1] > 1 and (plan[1] - 1) * units < k // 64
                    assert -(-rows // tm) * -(-n // tn) * plan[1] <= 256
                assert ops.wide_gated_form(rows, n, k) in (None, *range(len(ops.WIDE_FORMS)))
        assert ops.wide_split_plan(512, 4096, 12288) == (2, 4) and ops.wide_split_plan(256, 2560, 9728) == (4, 6)
        assert ops.wide_split_plan(2048, 4096, 4096) is None and ops.wide_split_plan(1500, 1024, 2048) is None
        assert ops.wide_gated_form(2048, 12288, 4096) == 0 and ops.wide_gated_form(512, 12288, 4096) == 1
    finally:
        for cached in (ops._wide_plan, ops.wide_split_plan, ops.wide_gated_form):
            cached.cache_clear()


def test_partial_sums_are_not_made_in_tiles_whose_way_out_is_slow():
    """5,120 outputs of K = 25,600: 1,152 rows in two ranges of tiles of 192 x 256 were slower than the whole product."""
    plans = {(rows, n, k): ops.wide_split_plan(rows, n, k) for rows in range(129, 2049) for n, k in ((5120, 25600), (5120, 17408), (4096, 12288), (2560, 9728))}
    assert all(plan is None or ops.WIDE_FORMS[plan[0]][:2] != (192, 256) for plan in plans.values())
    assert [plans[n, 5120, 25600] for n in (1034, 1152)] == [None, (0, 2)] and plans[513, 5120, 17408] == (0, 4)


def test_gated_products_whose_last_round_gives_a_compute_unit_two_tiles():
    """17,408 gated outputs of K = 5,120, 353 to 384 rows in 816 tiles of 128 x 128, two to a compute unit: the 304 beyond a round take nearly as long as
    512, and the product with the activation after it less.  Where the last round is nearly full, or the tile far ahead, the rule stays."""
    forms = {(rows, n, k): ops.wide_gated_form(rows, n, k) for rows in range(129, 2049) for n, k in ((17408, 5120), (12288, 4096), (9728, 2560), (3072, 1024))}
    assert all(forms[rows, 17408, 5120] is None for rows in range(257, 442)) and forms[442, 17408, 5120] == forms[256, 17408, 5120] == 1
    assert all(forms[rows, 12288, 4096] == 5 for rows in range(603, 641)) and forms[602, 12288, 4096] is None  # 448 of 512
    assert forms[384, 9728, 2560] == 5 and forms[768, 3072, 1024] == 5 and forms[640, 3072, 1024] == 4  # 456 of 512; 288, but 18 of 22 us


class Library:
    """The library's entry points and what runs, without a GPU: every shape has three candidates, whose kernels have the numbers 10 to 12, and
    takes a fourth one on; times[candidate] is what a run takes (9 where none is given)."""

    def __init__(self, monkeypatch, times=()):
        self.ran, self.times, self.adopted = [], dict(times), {}
        doors = {"as_blas_plan": lambda *shape: 3, "as_blas_candidate_index": lambda M, N, K, dtype, size, place: 10 + place,
                 "as_blas_adopt": self.adopt, "as_gemm_bf16_wide": None}  # fmt: skip
        monkeypatch.setattr(ops, "entry", doors.__getitem__)
        monkeypatch.setattr(ops, "_library_workspace", lambda device: torch.empty(1))
        monkeypatch.setattr(ops, "_library_call", lambda a, w, out, M, N, K, candidate: self.ran.append((M, candidate)))
        monkeypatch.setattr(ops, "_trial_run", self.trial_run)
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda: type("S", (), {"synchronize": lambda self: None})())

    def adopt(self, M, N, K, dtype, size, index):
        self.adopted[M] = index
        return index - 10

    def trial_run(self, trial, a, w, out, M, N, K):
        candidate = trial["ids"][len(trial["runs"]) % trial["count"]]
        self.ran.append((M, candidate))
        trial["runs"].append((candidate, Mark(), Mark(self.times.get(candidate, 9.0))))


class Matrix:
    """A matrix of bf16 as the dispatch looks at it, starting at a place of its choice."""

    def __init__(self, rows, columns, at=0):
        self.shape, self.dtype, self.at, self.device, self.is_cuda = (rows, columns), BF16, at, "cuda:0", True

    def data_ptr(self):
        return self.at


def settled(choices, M, N, K, run=None):
    """Runs the product of M rows until its trial has ended."""
    choices.tune_rows(M)
    run = run or (lambda: choices.gemm(Matrix(M, K), Matrix(N, K), Matrix(M, N), M, N, K))
    run()
    choices.settle()


def test_where_the_large_tile_is_no_candidate_the_trials_best_of_the_library_runs(monkeypatch):
    """A row count that follows a tuned one on which the large tile won takes the tile where it may win there too, and the library's fastest
    of that trial elsewhere; so do matrices that the tile does not take.  Not the library's first, which no trial has named."""
    library = Library(monkeypatch, {0: 8.0, 1: 5.0, 2: 4.0, ops.WIDE_CANDIDATE: 3.0})
    choices, N, K, tuned = ops.ProductChoices(), 4096, 4096, 1536
    settled(choices, tuned, N, K)
    assert choices.chosen() == {(tuned, N, K, BF16): ops.WIDE_CANDIDATE}
    asked = range(1025, tuned)
    without = [M for M in asked if not ops._own_candidates(M, N, K, BF16, None)]
    assert 1100 in without and 1520 not in without

    def runs(M, at=0):
        library.ran.clear()
        choices.gemm(Matrix(M, K, at), Matrix(N, K), Matrix(M, N), M, N, K)
        return library.ran

    for M in (1025, 1100, 1504, 1505, 1520):
        for _ in range(2):
            assert runs(M) == [(M, 2 if M in without else ops.WIDE_CANDIDATE)]
        assert library.adopted.get(M) == (12 if M in without else None)
    assert runs(1520, at=8) == [(1520, 2)] and library.adopted[1520] == 12 and runs(1520) == [(1520, ops.WIDE_CANDIDATE)]
    assert runs(tuned, at=8) == [(tuned, 2)] and runs(tuned) == [(tuned, ops.WIDE_CANDIDATE)]
    door = ops.entry
    monkeypatch.setattr(ops, "entry", lambda name: (lambda *shape: -1) if name == "as_blas_adopt" else door(name))
    assert runs(1101) == [(1101, 0)]  # a shape that does not take that kernel on: its own first


def user(monkeypatch, library, choices, N, K, gated=False):
    """One product of M rows as a layer makes it: down in parts where that pays, else whole; or gate and up with their activation."""
    for name in ("_check", "silu_mul", "_few_rows", "_tile_rows"):
        monkeypatch.setattr(ops, name, lambda *args, **kw: None)
    monkeypatch.setattr(ops, "_ptr", lambda t: 0)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "call", lambda name, *args: library.ran.append((args[3], name)))
    w = Matrix(N, K)

    def product(M):
        library.ran.clear()
        a, out = Matrix(M, K), Matrix(M, N // 2 if gated else N)
        if gated:
            a.device = "meta"  # gate and up stand there
            ops.gemm_silu_mul(a, w, out, choices)
        else:
            a.device = "meta"  # the sums stand there
            if ops.gemm_split_sums(a, w, choices) is None:
                ops.gemm(a, w, out, choices)
        return library.ran

    return product


PROMPT_LENGTHS = [n for p in range(7, 12) for n in (2**p, 3 * 2 ** (p - 1)) if n <= 2048]  # what a warm-up runs up to 2,048 tokens


@pytest.mark.parametrize("N,K,gated,away", [(4096, 12288, False, 413), (5120, 17408, False, 165), (34816, 5120, True, 542), (24576, 4096, True, 162)])
def test_row_counts_on_the_librarys_side_of_a_rule_find_a_settled_one(monkeypatch, N, K, gated, away):
    """The rules that give a product of many rows to the large tile say yes and no by row count, the warm-up knows a few counts: those that take the
    tile try the library's candidates too, for the counts below them that do not."""
    library = Library(monkeypatch, {0: 8.0, 1: 5.0, 2: 4.0})
    choices = ops.ProductChoices()
    product = user(monkeypatch, library, choices, N, K, gated)
    tile = (lambda M: ops.wide_gated_form(M, N // 2, K)) if gated else (lambda M: ops.wide_split_plan(M, N, K))
    for M in PROMPT_LENGTHS[1:]:
        choices.tune_rows(M)
        product(M)
        assert choices.trials_pending()
        choices.settle()
        assert product(M) == [(M, "as_gemm_bf16_wide" if tile(M) is not None else 2)]
    fell = 0
    for M in range(129, 2049):
        if M not in choices.tuned_rows and tile(M) is None:
            above = min(m for m in PROMPT_LENGTHS if m >= M)
            fell += tile(above) is not None
            assert product(M) == [(M, 2)] and library.adopted[M] == 12
    assert fell == away
    fixed = ops.ProductChoices(fixed=True)  # no trials: the rule
    fixed.tune_rows(1024)
    assert user(monkeypatch, library, fixed, N, K, gated)(1024) == [(1024, "as_gemm_bf16_wide")] and not fixed.trials_pending()


@pytest.mark.parametrize("N,K,gated", [(6144, 0, True), (0, 1024, True), (3072, 0, False), (0, 1024, False)])
def test_products_without_columns_or_outputs_are_not_the_large_tiles(monkeypatch, N, K, gated):
    """A sum of nothing is zero and no outputs are none, as torch's product gives them; the large tile refuses both."""
    library = Library(monkeypatch)
    assert user(monkeypatch, library, ops.ProductChoices(), N, K, gated)(300) == [(300, 0)]


@pytest.mark.parametrize("H,KV,D,rows,context,change,how", [
    (16, 8, 128, 4, 600, None, "one"), (16, 8, 128, 32, 200, None, "one"), (16, 8, 128, 33, 200, None, "one"),  # 8 workgroups a row
    (16, 8, 128, 8, 500, None, "one"), (16, 8, 128, 1, 2000, None, "one"), (16, 8, 128, 8, 2000, None, "one"),  # contexts in parts
    (16, 8, 64, 33, 200, None, "one"), (8, 2, 64, 64, 6000, None, "one"), (16, 8, 128, 4, 600, "q gains elsewhere", "two"),
    (16, 8, 128, 4, 600, "k gains elsewhere", "two"), (16, 8, 128, 4, 600, "no norm", "two"), (16, 8, 128, 4, 600, "no rotation", "two"),
    (16, 8, 128, 4, 600, "half of a head turned", "two"), (16, 8, 96, 4, 600, None, "two"), (16, 8, 128, 4, 600, "a prompt", "two"),
    (16, 8, 128, 4, 600, "pages of 8", "two"), (16, 8, 128, 64, 8000, "bf16", "bf16"),
])  # fmt: skip
def test_the_route_of_a_32_bit_decode_step(monkeypatch, H, KV, D, rows, context, change, how):
    """Norm, rotation, store and attention in one kernel at every number of rows and tokens, for the heads, norms, rotations and pages that it
    takes and gains that start on 16 bytes; else in two."""
    from types import SimpleNamespace

    from atomserve_amd.parts.attention import Attention

    made, dtype = [], BF16 if change == "bf16" else F32
    for name, word in (("attn_f32_fresh", "one"), ("attn_decode_fresh", "bf16"), ("qk_norm_rope_store", "two"), ("gemm", None)):
        monkeypatch.setattr(ops, name, lambda *args, word=word, **kw: made.append(word))
    gains = [torch.empty(D + 4)[(1 if change == f"{n} gains elsewhere" else 0) :][:D] for n in "qk"]
    turned = None if change == "no rotation" else torch.empty(rows, D // (4 if change == "half of a head turned" else 2), 2)
    mixer = SimpleNamespace(
        spec=SimpleNamespace(num_heads=H, num_kv_heads=KV, head_dim=D, hidden_size=64, window=0, scale=1.0,
                             qk_norm=None if change == "no norm" else SimpleNamespace(eps=1e-6)),
        env=SimpleNamespace(dtype=dtype, products=None), qkv=None, o=None, position=SimpleNamespace(prepare=lambda step: turned),
        q_norm_weight=gains[0], k_norm_weight=gains[1], attend=lambda *args: None)  # fmt: skip
    step = SimpleNamespace(decode_only=change != "a prompt", max_context=context, positions=None, all_tokens=None)
    cache = SimpleNamespace(block_size=8 if change == "pages of 8" else 16, slots=None, writes=True, k_pages=None, v_pages=None, block_tables=None)
    Attention.forward(mixer, torch.empty(rows, 64, dtype=dtype), step, cache)
    assert [word for word in made if word] == [how]


@pytest.mark.parametrize("budget,lengths", [(127, []), (128, [128]), (200, [128, 192, 200]), (512, [128, 192, 256, 384, 512]), (600, [128, 192, 256, 384, 512, 600])])
def test_a_warm_up_tries_the_steps_budget_itself(monkeypatch, budget, lengths):
    """A budget is a tuned row count wherever it lies: its trials belong to the warm-up, not to the first steps that fill it."""
    from types import SimpleNamespace

    from atomserve_amd.engine.runner import ModelRunner

    monkeypatch.setattr(ops, "prepare_library_adoption", lambda: True)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    products, ran = ops.ProductChoices(), []
    runner = SimpleNamespace(model=SimpleNamespace(env=SimpleNamespace(products=products)), device=torch.device("cuda"),
                             manager=SimpleNamespace(block_size=16, state_groups=[], paged_groups=[0]), vocab_size=150, step=lambda rows: ran.append(rows[0].tokens))  # fmt: skip
    assert ModelRunner.tune_prompt_lengths(runner, budget) == lengths == [len(tokens) for tokens in ran]
    assert all(len(set(tokens)) == min(len(tokens), 150) and 0 <= min(tokens) <= max(tokens) < 150 for tokens in ran)  # not one token again and again
    assert set(lengths) <= products.tuned_rows


@pytest.mark.parametrize("ends_after,passes", [(1, [1, 1, 1]), (3, [3, 3, 3]), (9, [4, 4, 9]), (500, [4, 4, 73])])
def test_the_budgets_trials_run_inside_passes(monkeypatch, ends_after, passes):
    """A model of few layers needs many passes until every candidate has run; the other lengths' trials are ended by `settle` after four."""
    from types import SimpleNamespace

    from atomserve_amd.engine.runner import ModelRunner

    monkeypatch.setattr(ops, "prepare_library_adoption", lambda: True)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    ran, settled_at = [], []
    products = SimpleNamespace(fixed=False, tune_rows=lambda n: ran.append(0), trials_pending=lambda: ran[-1] < ends_after, settle=lambda: settled_at.append(ran[-1]))
    runner = SimpleNamespace(model=SimpleNamespace(env=SimpleNamespace(products=products)), device=torch.device("cuda"), vocab_size=150,
                             manager=SimpleNamespace(block_size=16, state_groups=[], paged_groups=[0]), step=lambda rows: ran.append(ran.pop() + 1))  # fmt: skip
    ModelRunner.tune_prompt_lengths(runner, 200)
    assert ran == settled_at == passes
