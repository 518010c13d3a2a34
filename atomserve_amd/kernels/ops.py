"""One checked Python wrapper per HIP kernel.

Each wrapper verifies on the host what the kernel and its grid assume (device, dtype,
contiguity, shapes) and only then launches on torch's current stream.  Nothing here
computes with torch operators: if a library is missing the call raises.
"""

import functools
import math

import torch

from atomserve_amd.kernels.lib import KernelError, call, entry, watch

F32, BF16, I32 = torch.float32, torch.bfloat16, torch.int32
_DT = {F32: 0, BF16: 1}


def _stream() -> int:
    """The raw handle of torch's current stream on the current device (an eager step makes some
    hundred launches, so this asks the binding directly instead of building a Stream object)."""
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _check(t, name, dtype=None, shape=None):
    """Runs before every launch, several times: written for the case that all is well."""
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise KernelError(f"{name} must be a tensor on the GPU")
    if not t.is_contiguous():
        raise KernelError(f"{name} must be contiguous")
    if dtype is not None and t.dtype is not dtype and (isinstance(dtype, torch.dtype) or t.dtype not in dtype):
        raise KernelError(f"{name} has dtype {t.dtype}, expected {dtype}")
    if shape is not None:
        have = t.shape
        good = len(have) == len(shape)
        if good:
            for d, s in zip(have, shape):
                if s is not None and d != s:
                    good = False
                    break
        if not good:
            raise KernelError(f"{name} has shape {tuple(have)}, expected {tuple(shape)}")


def _ptr(t) -> int:
    if t is None:
        return 0
    if watch.held is not None:
        watch.held.append(t)
    return t.data_ptr()


# ---- weights in the order in which a wave reads them -------------------------------------------
#
# The few-rows and tile products stream a weight matrix once per step.  `Streamed(w)` holds a bf16
# matrix [R, K] (R % 16 == 0, K % 64 == 0) a second time, its 16-byte pieces lying as a wave of those
# kernels takes them; the products that are handed the `Streamed` read that copy (every load
# instruction 1 KB in one piece, marked as not to be kept: 7 per cent less time for the 144 products of
# a decode step at Qwen3-8B sizes), the library's products and everything else read the rows.  The
# owner of the matrix (a part, the decoder for its head) owns the `Streamed` and with it the copy's
# memory; whoever changes the rows in place afterwards calls `refresh()`.


class Streamed:
    """A weight matrix as the products of this module read it: `rows`, the tensor [R, K] itself, and
    `wave`, its copy in wave order, or None where the dtype or the sizes do not allow one or the owner
    asked for none (`copy=False`: the copy's bytes are saved, decode steps stream the rows)."""

    __slots__ = ("rows", "wave")

    def __init__(self, rows, copy: bool = True):
        self.rows, self.wave = rows, None
        if copy:
            self.refresh()

    @staticmethod
    def possible(w) -> bool:
        return w.dtype == BF16 and w.dim() == 2 and w.is_cuda and w.is_contiguous() and w.shape[0] % 16 == 0 and w.shape[1] % 64 == 0

    def refresh(self):
        """Makes the copy (anew) from the rows as they are now; returns it, None where there can be none."""
        if not self.possible(self.rows):
            self.wave = None
            return None
        if self.wave is None:
            self.wave = torch.empty_like(self.rows)
        call("as_wave_order", _ptr(self.rows), _ptr(self.wave), self.rows.shape[0], self.rows.shape[1], _stream())
        return self.wave

    @property
    def wave_bytes(self) -> int:
        return 0 if self.wave is None else self.wave.numel() * self.wave.element_size()


def _rows(w):
    """The matrix itself of what a product was handed as its weights (a tensor, or a `Streamed`)."""
    return w.rows if isinstance(w, Streamed) else w


def _wave_ptr(w) -> int:
    """The address of the copy in wave order of a product's weights, 0 if they have none."""
    if isinstance(w, Streamed) and w.wave is not None:
        return w.wave.data_ptr()
    return 0


def embed_gather(table, ids, out, scale: float = 1.0) -> None:
    """out[t] = scale * table[ids[t]] as fp32.  table [V, h] fp32|bf16, ids [T] int32, out [T, h] fp32."""
    _check(table, "table", (F32, BF16), (None, None))
    vocab, width = table.shape
    _check(ids, "ids", I32, (None,))
    _check(out, "out", F32, (ids.shape[0], width))
    call("as_embed_gather", _ptr(table), _DT[table.dtype], _ptr(ids), _ptr(out), ids.shape[0], width, vocab,
         float(scale), _stream())  # fmt: skip


def logits_finish(logits, scale: float = 1.0, softcap: float = 0.0) -> None:
    """logits = softcap * tanh(scale * logits / softcap) in place (softcap 0: the scale alone); fp32."""
    _check(logits, "logits", F32)
    if softcap < 0:
        raise KernelError("a soft cap of logits is positive, or 0 for none")
    call("as_logits_finish", _ptr(logits), logits.numel(), float(scale), float(softcap), _stream())


def rmsnorm(x, weight, eps, out, delta=None, rows=None, update_x=True, split_sums=None) -> None:
    """out[r] = norm(x[s] + delta[s]) * weight with s = rows[r] (or r); x fp32 [T, n] gets the
    sum written back when `delta` is given and `update_x`.  out, delta: fp32|bf16.
    split_sums: instead of `delta`, the fp32 partial sums [splits, T, n] of the product that makes it
    (`gemm_split`); they are added up and rounded to out's dtype as the product would have been."""
    _check(x, "x", F32, (None, None))
    T, n = x.shape
    _check(weight, "weight", (F32, BF16), (n,))
    n_out = T
    if rows is not None:
        _check(rows, "rows", I32, (None,))
        n_out = rows.shape[0]
    _check(out, "out", (F32, BF16), (n_out, n))
    if delta is not None:
        _check(delta, "delta", out.dtype, (T, n))
    if out.dtype == F32 and weight.dtype != F32:
        raise KernelError("fp32 norm needs an fp32 weight")
    if split_sums is not None:
        if delta is not None:
            raise KernelError("a pending sum comes as one tensor or as partial sums, not both")
        _check(split_sums, "split_sums", F32, (None, T, n))
        call("as_rmsnorm_split", _ptr(x), _ptr(split_sums), split_sums.shape[0], T, _ptr(rows), _ptr(weight),
             _DT[weight.dtype], float(eps), _ptr(out), _DT[out.dtype], n_out, n, int(bool(update_x)), _stream())  # fmt: skip
        return
    call("as_rmsnorm", _ptr(x), _ptr(delta), _ptr(rows), _ptr(weight), _DT[weight.dtype], float(eps), _ptr(out),
         _DT[out.dtype], n_out, n, int(bool(update_x)), _stream())  # fmt: skip


def rope_table(positions, inv_freq, out, magnitude: float = 1.0) -> None:
    """out[t, i] = magnitude * (cos, sin)(positions[t] * inv_freq[i]); inv_freq fp64 [R/2], out fp32 [T, R/2, 2]."""
    _check(positions, "positions", I32, (None,))
    _check(inv_freq, "inv_freq", torch.float64, (None,))
    _check(out, "out", F32, (positions.shape[0], inv_freq.shape[0], 2))
    if magnitude == 1.0:
        call("as_rope_table", _ptr(positions), _ptr(inv_freq), _ptr(out), positions.shape[0], inv_freq.shape[0], _stream())
    else:
        call("as_rope_table_scaled", _ptr(positions), _ptr(inv_freq), _ptr(out), positions.shape[0], inv_freq.shape[0],
             float(magnitude), _stream())  # fmt: skip


def qk_norm_rope_store(qkv, q_weight, k_weight, cos_sin, slots, q_out, k_pages, v_pages, num_heads,
                       num_kv_heads, eps, store_kv=True) -> None:  # fmt: skip
    """Per-head norm (if weights are given), rotation (if `cos_sin` is given) and the cache store.

    qkv [T, H + 2 KV, D]; q_out [T, H, D]; k_pages [num_pages, KV, block_size, D], v_pages
    [num_pages, KV, D, block_size] (values transposed within a page); slots [T] int32
    (page * block_size + offset, or -1 for a token whose keys are not stored)."""
    _check(qkv, "qkv", (F32, BF16), (None, num_heads + 2 * num_kv_heads, None))
    T, _, D = qkv.shape
    _check(q_out, "q_out", qkv.dtype, (T, num_heads, D))
    R = 0
    if cos_sin is not None:
        _check(cos_sin, "cos_sin", F32, (T, None, 2))
        R = 2 * cos_sin.shape[1]
        if R > D:
            raise KernelError(f"rotary width {R} exceeds head width {D}")
    w_dtype = qkv.dtype
    if q_weight is not None:
        _check(q_weight, "q_weight", (F32, BF16), (D,))
        _check(k_weight, "k_weight", q_weight.dtype, (D,))
        w_dtype = q_weight.dtype
        if qkv.dtype == F32 and w_dtype != F32:
            raise KernelError("fp32 q/k norm needs fp32 weights")
    elif k_weight is not None:
        raise KernelError("q and k norm weights come together")
    block_size = 1
    if store_kv:
        _check(slots, "slots", I32, (T,))
        _check(k_pages, "k_pages", qkv.dtype, (None, num_kv_heads, None, D))
        block_size = k_pages.shape[2]
        _check(v_pages, "v_pages", qkv.dtype, (k_pages.shape[0], num_kv_heads, D, block_size))
    call("as_qk_norm_rope_store", _ptr(qkv), _DT[qkv.dtype], _ptr(q_weight), _ptr(k_weight), _DT[w_dtype],
         _ptr(cos_sin), _ptr(slots) if store_kv else 0, _ptr(q_out), _ptr(k_pages) if store_kv else 0,
         _ptr(v_pages) if store_kv else 0, T, num_heads, num_kv_heads, D, R, float(eps), block_size,
         int(bool(store_kv)), _stream())  # fmt: skip


def silu_mul(gate_up, out) -> None:
    """out[t, i] = silu(gate_up[t, i]) * gate_up[t, I + i]."""
    _check(gate_up, "gate_up", (F32, BF16), (None, None))
    T, two_i = gate_up.shape
    if two_i % 2:
        raise KernelError("gate_up needs an even width")
    _check(out, "out", gate_up.dtype, (T, two_i // 2))
    call("as_silu_mul", _ptr(gate_up), _ptr(out), _DT[gate_up.dtype], T, two_i // 2, _stream())


SINGLE_QUERY_MAX_HEAD_DIM = 256


def _sight(window, keep_first, chunk, softcap, sink, q, out) -> tuple:
    """(window, keep, chunk, cap, sink, sinks, wide) as the attention kernels take them: what a query sees, how scores become
    weights and whether bfloat16 heads' results are written in fp32."""
    _check(out, "out", (q.dtype, F32), tuple(q.shape))
    if window < 0 or keep_first < 0 or softcap < 0 or chunk < 0 or (chunk and window):
        raise KernelError("attention: a window, a number of kept tokens, a cap of the scores and a chunk are not negative; "
                          "a sequence is cut into chunks or seen through a window")  # fmt: skip
    sinks = 0
    if isinstance(sink, torch.Tensor):
        _check(sink, "sinks", F32, (q.shape[1],))
        sinks = _ptr(sink)
    has_sink = 1 if sinks else int(bool(sink))
    return int(window), int(keep_first) if window > 0 else 0, int(chunk), float(softcap), has_sink, sinks, int(out.dtype != q.dtype)


def attn_single_query(q, k_pages, v_pages, items, positions, tok_row, block_tables, out, scale, window,
                      max_context, part_size=None, force_generic=False, keep_first=0, softcap=0.0, sink=False, chunk=0) -> None:  # fmt: skip
    """Attention of single query tokens over the paged cache.  bfloat16 with head widths in steps
    of 32 and pages of a multiple of 16 tokens runs on the matrix cores (a group of more than 16 query
    heads, or of wide heads that overfill a workgroup's LDS, as several equal groups that read the same kv
    head), and so do the fp32 heads that `attn_f32_supported` names, in 32 bits; everything else on the general kernel.

    q, out [T, H, D] (out fp32 for bfloat16 heads: the results unrounded); items [N] int32: the tokens (rows of q) to process, None for all of them in
    order; positions, tok_row [T] int32 (tok_row None: token t belongs to row t, a decode step);
    block_tables [R, W] int32; max_context: host bound on positions[items] + 1.
    window > 0: a query at p sees the keys p - window + 1 .. p and those of the first `keep_first` positions.
    chunk > 0 (without a window): a query sees the keys of its own chunk, chunks of that many positions counted from 0.
    softcap > 0: a score s counts as softcap tanh(s / softcap).  sink: the softmax's denominator has one more score, of 0
    (True) or per query head (a tensor fp32 [H])."""
    _check(q, "q", (F32, BF16), (None, None, None))
    T, H, D = q.shape
    sight = _sight(window, keep_first, chunk, softcap, sink, q, out)
    _check(k_pages, "k_pages", q.dtype, (None, None, None, D))
    _, KV, bs, _ = k_pages.shape
    _check(v_pages, "v_pages", q.dtype, (k_pages.shape[0], KV, D, bs))
    if items is not None:
        _check(items, "items", I32, (None,))
    _check(positions, "positions", I32, (T,))
    if tok_row is not None:
        _check(tok_row, "tok_row", I32, (T,))
    _check(block_tables, "block_tables", I32, (None, None))
    if tok_row is None and block_tables.shape[0] < T:
        raise KernelError(f"attention: {T} tokens that are their own rows need as many block tables")
    N = T if items is None else items.shape[0]
    if N == 0:
        return
    piece = 4 if q.dtype == F32 else 8
    if H % KV or D % piece or D > SINGLE_QUERY_MAX_HEAD_DIM:
        raise KernelError(f"attention: unsupported heads {H}/{KV} or head width {D} "
                          f"(needs a multiple of {piece}, at most {SINGLE_QUERY_MAX_HEAD_DIM})")  # fmt: skip
    if max_context > block_tables.shape[1] * bs:
        raise KernelError("attention: block tables are shorter than the longest context")
    share = 0 if force_generic else _decode_mfma_share(q.dtype, H, KV, D, bs)
    mfma = share > 0
    if share > 1:
        part_size, P, part_m, part_l, part_acc = _partitions(N, H, KV * share, D, max_context, window or chunk, True, part_size, q.device, sight[1])
        call("as_attn_decode_mfma_shared", _ptr(q), _ptr(k_pages), _ptr(v_pages), _ptr(items), N, _ptr(positions),
             _ptr(tok_row), _ptr(block_tables), block_tables.shape[1], _ptr(out), _ptr(part_m), _ptr(part_l),
             _ptr(part_acc), H, KV * share, D, bs, float(scale), *sight, part_size, P, share, _stream())  # fmt: skip
        return
    matrix32 = not force_generic and attn_f32_supported(q.dtype, H, KV, D, bs, sight[1]) and (part_size is None or part_size % 32 == 0)
    part_size, P, part_m, part_l, part_acc = _partitions(N, H, KV, D, max_context, window or chunk, mfma or matrix32, part_size, q.device, sight[1])
    if matrix32:
        call("as_attn_f32", _ptr(q), _ptr(k_pages), _ptr(v_pages), 0, 0, 0, _ptr(items), N, _ptr(positions), _ptr(tok_row),
             _ptr(block_tables), block_tables.shape[1], _ptr(out), _ptr(part_m), _ptr(part_l), _ptr(part_acc), H, KV, D, bs,
             float(scale), *sight, part_size, P, _stream())  # fmt: skip
        return
    if mfma:
        call("as_attn_decode_mfma", _ptr(q), _ptr(k_pages), _ptr(v_pages), _ptr(items), N, _ptr(positions),
             _ptr(tok_row), _ptr(block_tables), block_tables.shape[1], _ptr(out), _ptr(part_m), _ptr(part_l),
             _ptr(part_acc), H, KV, D, bs, float(scale), *sight, part_size, P, _stream())  # fmt: skip
        return
    call("as_attn_single_query", _ptr(q), _ptr(k_pages), _ptr(v_pages), _DT[q.dtype], _ptr(items), N,
         _ptr(positions), _ptr(tok_row), _ptr(block_tables), block_tables.shape[1], _ptr(out), _ptr(part_m),
         _ptr(part_l), _ptr(part_acc), H, KV, D, bs, float(scale), *sight, part_size, P, _stream())  # fmt: skip


def _decode_mfma_share(dtype, H: int, KV: int, D: int, bs: int) -> int:
    """Into how many equal groups the query heads of a kv head are cut for the bf16 matrix-core kernel of single queries (whose
    workgroup holds a group of up to 16); 0 where another kernel runs."""
    if dtype != BF16 or D % 32 or bs % 16:
        return 0
    G = H // KV
    return next((G // g for g in range(min(G, 16), 0, -1) if G % g == 0 and _decode_mfma_fits(D, g)), 0)


def contexts_cut(rows: int, H: int, KV: int, D: int, dtype, bs: int, context: int, window: int = 0, keep_first: int = 0) -> bool:
    """Whether `attn_single_query` (and `attn_decode_fresh`) cuts contexts of up to `context` keys into partitions that another
    kernel merges, for a decode step of `rows` rows."""
    share = _decode_mfma_share(dtype, H, KV, D, bs)
    matrix = share > 0 or attn_f32_supported(dtype, H, KV, D, bs, keep_first)
    return _partitions(rows, H, KV * max(1, share), D, context, window, matrix, None, "meta", keep_first)[1] > 1


def attn_f32_supported(dtype, num_heads: int, num_kv_heads: int, head_dim: int, block_size: int, keep_first: int = 0) -> bool:
    """Whether 32-bit heads run on the matrix cores (`attn_f32`, products and sums in 32 bits): heads of 64 or 128, at most 16 of
    them to a kv head, whole steps of 16 keys to a page, no kept first keys; the rest runs on the general kernel."""
    return (dtype == F32 and head_dim in (64, 128) and num_heads % num_kv_heads == 0 and num_heads // num_kv_heads <= 16
            and block_size % 16 == 0 and keep_first == 0)  # fmt: skip


# What 32-bit attention costs (microseconds, fitted to the kernel's times for portions of 9 to 512 tokens behind 0 to 30,000 keys, 4 to
# 16 heads on 1 to 8 kv heads), by head width: (a prompt tile's launch and merge, 64 keys of one, a single query's launch,
# a microsecond of `_partition_cost`).
F32_ATTENTION_COSTS = {64: (5.2, 1.07, 4.0, 1.2), 128: (7.8, 1.65, 4.5, 2.2)}


def attn_tiles_preferred(tokens: int, short: int, H: int, KV: int, D: int, max_context: int, window: int) -> bool:
    """Whether a step of 32-bit heads runs its long rows as prompt tiles (`attn_prefill_f32`, the `short` tokens of short rows
    beside them as single queries) or all of its tokens as single queries.  A tile reads its keys once for all of its queries,
    but walks all of them in one workgroup; single queries' keys are cut into partitions.  16 heads of 128 on 8 kv heads,
    tiles against single queries: 9 tokens alone 9.3 and 6.6 us, 64 10.5 and 8.8; 9 behind 2,000 keys 61 and 35, 33 61 and 81;
    9 behind 8,000 209 and 97, 64 213 and 350; 9 behind 30,000 760 and 315."""
    base, step, one, by = F32_ATTENTION_COSTS[D]
    span = _seen_keys(max_context, window, 0, True)

    def single(n: int) -> float:
        groups = n * KV
        if groups >= attn_fill_groups():
            return one + by * (_partition_cost(groups, span, _up32(span)) - 4.0)
        return one + by * (min(_partition_cost(groups, span, part) for part in MFMA_PARTITIONS) - 4.0)

    workgroups = (tokens - short) * H / 16  # two share a compute unit, and 512 take 1.76 times as long as 256
    tiles = (base + step * max(1.0, span / 64)) * max(1.0, workgroups / (1.13 * compute_units()))
    return tiles + (single(short) if short else 0.0) <= single(tokens)


def attn_prefill_f32(q, k_pages, v_pages, tiles, block_tables, out, scale, window, max_context, softcap=0.0, sink=False, chunk=0) -> None:
    """`attn_prefill` for the 32-bit heads that `attn_f32_supported` names (tiles of up to PREFILL_TILE_QUERIES tokens)."""
    _check(q, "q", F32, (None, None, None))
    T, H, D = q.shape
    sight = _sight(window, 0, chunk, softcap, sink, q, out)
    _check(k_pages, "k_pages", F32, (None, None, None, D))
    _, KV, bs, _ = k_pages.shape
    _check(v_pages, "v_pages", F32, (k_pages.shape[0], KV, D, bs))
    _check(tiles, "tiles", I32, (None, 4))
    _check(block_tables, "block_tables", I32, (None, None))
    if tiles.shape[0] == 0:
        return
    if not attn_f32_supported(q.dtype, H, KV, D, bs):
        raise KernelError(f"prefill attention: unsupported heads {H}/{KV}, head width {D} or page size {bs}")
    if max_context > block_tables.shape[1] * bs:
        raise KernelError("attention: block tables are shorter than the longest context")
    call("as_attn_f32", _ptr(q), _ptr(k_pages), _ptr(v_pages), _ptr(tiles), tiles.shape[0], PREFILL_TILE_QUERIES, 0, 0, 0, 0,
         _ptr(block_tables), block_tables.shape[1], _ptr(out), 0, 0, 0, H, KV, D, bs, float(scale), *sight, 16, 1, _stream())  # fmt: skip


DECODE_MFMA_MAX_LDS = 64 << 10  # what a workgroup may ask for without raising the kernel's limit


def compute_units() -> int:
    """Compute units of the current GPU (256 on an MI355X); grids and the fitted costs below scale with it."""
    global _compute_units
    if _compute_units is None:
        _compute_units = torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
    return _compute_units


_compute_units = None


def _decode_mfma_fits(head_dim: int, group: int) -> bool:
    """Whether the matrix-core decode kernel's workgroup (queries of a group and four partial outputs
    in LDS) stays within the LDS a kernel gets unasked; wide heads in large groups do not."""
    return 4 * (128 + 4 * head_dim * group) + 1024 <= DECODE_MFMA_MAX_LDS


def attn_fill_groups() -> int:
    """(token, kv head) pairs from which on whole contexts beat partitions and their merge: one and a
    half per compute unit (measured on 256)."""
    return compute_units() * 3 // 2


MFMA_PARTITIONS = (128, 256, 512, 1024, 2048)  # keys per workgroup of the matrix-core decode kernel


# Microseconds of the merge's kernel beside what `_partition_cost` counts; whole contexts have none (16 heads on 8 kv heads, 1 request:
# 100 keys 7.5 us whole and 10.9 in partitions of 128 with the merge, 256 keys 9.5 and 10.8, 400 keys 12.7 and 10.2).
MERGE_LAUNCH = 4.1


def _partition_cost(groups: int, span: int, part: int) -> float:
    """Microseconds, roughly, of the decode attention and its merge when `groups` (token, kv head) pairs
    cut `span` keys into partitions of `part`: a workgroup costs 4 us and 25 ns a key, two of them run
    on a compute unit at a time, and the merge 0.6 us a partition.  Fitted to the kernel's times at 1
    to 32 requests of 500 to 33,000 keys (heads of 128, 8 kv heads, 256 compute units); what it picks
    is within 2 per cent of the best partition size on average there, where one size for all was 8 per
    cent off."""
    parts = math.ceil(span / part)
    return (4.0 + 0.025 * min(part, span)) * max(1.0, groups * parts / (2 * compute_units())) + 0.6 * parts


def _up32(n: int) -> int:
    return -(-n // 32) * 32


def _seen_keys(max_context: int, window: int, keep_first: int, mfma: bool) -> int:
    """The most keys that a query of these contexts walks: with a window those of the window and the kept first ones
    (the matrix-core kernel in whole steps of 32, and a window that starts within a step takes it whole)."""
    if window <= 0:
        return max_context
    if mfma:
        return min(_up32(max_context), _up32(window + 31) + _up32(keep_first))
    return min(max_context, window + keep_first)


def _partitions(N, H, KV, D, max_context, window, mfma, part_size, device, keep_first=0):
    """How the keys of N single queries are cut for the split-KV kernels, and the buffers of the
    partial results: (part_size, P, part_m, part_l, part_acc), the buffers None when P == 1.  What is cut is the
    list of the keys a query sees, in order: whole contexts, or the kept first keys and then the window's."""
    span = _seen_keys(max_context, window, keep_first, mfma)
    G = H // KV
    if part_size is None:
        # Enough partitions to occupy the GPU when few tokens are in the batch, few enough that
        # the merge stays small; boundaries are multiples of part_size in the list of visible keys.
        if mfma:
            groups = N * KV
            if groups >= attn_fill_groups():
                part_size = -(-span // 32) * 32  # enough workgroups without partitions: no merge
            else:
                part_size = min(MFMA_PARTITIONS, key=lambda part: _partition_cost(groups, span, part) + (MERGE_LAUNCH if part < span else 0.0))
        else:
            groups, part_size = N * KV * max(1, (G + 7) // 8), 256
            while part_size < span and groups * math.ceil(span / part_size) > 2048:
                part_size *= 2
    if mfma and part_size % 32:
        raise KernelError("attention: partitions of the matrix-core kernel are multiples of 32 keys")
    P = max(1, math.ceil(span / part_size))
    part_m = part_l = part_acc = None
    if P > 1:
        part_m = torch.empty((N, H, P), dtype=F32, device=device)
        part_l = torch.empty((N, H, P), dtype=F32, device=device)
        part_acc = torch.empty((N, H, P, D), dtype=F32, device=device)
    return part_size, P, part_m, part_l, part_acc


def attn_decode_fresh_supported(dtype, num_heads: int, num_kv_heads: int, head_dim: int, block_size: int,
                                rotary_dim: int, qk_norm: bool) -> bool:
    """Whether `attn_decode_fresh` takes this case: bfloat16 heads of 64, 128, 192 or 256 with a per-head
    norm, rotated whole, at most 16 query heads to a kv head, pages of a multiple of 16 tokens."""
    return (dtype == BF16 and head_dim % 64 == 0 and head_dim <= 256 and rotary_dim == head_dim and qk_norm
            and num_heads % num_kv_heads == 0 and num_heads // num_kv_heads <= 16 and block_size % 16 == 0
            and _decode_mfma_fits(head_dim, num_heads // num_kv_heads))  # fmt: skip


def attn_decode_fresh(qkv, q_weight, k_weight, cos_sin, slots, eps, store_kv, k_pages, v_pages, positions,
                      block_tables, out, num_heads, scale, window, max_context, part_size=None, order=None) -> None:
    """A decode step from the projection's output, in one kernel: what `qk_norm_rope_store` and then
    `attn_single_query` do for tokens that are their own rows (token t reads block table t).

    qkv [T, H + 2 KV, D] bf16; q_weight, k_weight [D] bf16 or fp32; cos_sin [T, D/2, 2] fp32;
    slots [T] int32; store_kv False: queries only, the pages already hold the tokens' keys and values
    (a run that reads another run's cache); out [T, H, D]; order [T] int32: the tokens in the order in
    which the workgroups take them (a permutation; longest contexts first keeps the compute units evenly
    busy when whole contexts are walked), None: as they come."""
    _check(qkv, "qkv", BF16, (None, None, None))
    T, heads, D = qkv.shape
    H = num_heads
    _check(k_pages, "k_pages", BF16, (None, None, None, D))
    _, KV, bs, _ = k_pages.shape
    if heads != H + 2 * KV:
        raise KernelError(f"qkv has {heads} heads, expected {H} + 2 x {KV}")
    _check(v_pages, "v_pages", BF16, (k_pages.shape[0], KV, D, bs))
    _check(out, "out", BF16, (T, H, D))
    _check(positions, "positions", I32, (T,))
    _check(block_tables, "block_tables", I32, (None, None))
    if block_tables.shape[0] < T:
        raise KernelError(f"attention: {T} tokens that are their own rows need as many block tables")
    R = 2 * cos_sin.shape[1] if cos_sin is not None else 0
    if not attn_decode_fresh_supported(BF16, H, KV, D, bs, R, q_weight is not None and k_weight is not None):
        raise KernelError(f"attention from fresh projections: unsupported heads {H}/{KV}, head width {D}, "
                          f"rotary width {R}, page size {bs}, or no per-head norm")  # fmt: skip
    _check(cos_sin, "cos_sin", F32, (T, D // 2, 2))
    _check(q_weight, "q_weight", (F32, BF16), (D,))
    _check(k_weight, "k_weight", q_weight.dtype, (D,))
    w_dtype = q_weight.dtype
    if store_kv:
        _check(slots, "slots", I32, (T,))
    if order is not None:
        _check(order, "order", I32, (T,))
    if T == 0:
        return
    if max_context > block_tables.shape[1] * bs:
        raise KernelError("attention: block tables are shorter than the longest context")
    part_size, P, part_m, part_l, part_acc = _partitions(T, H, KV, D, max_context, window, True, part_size, qkv.device)
    call("as_attn_decode_fresh", _ptr(qkv), _ptr(q_weight), _ptr(k_weight), _DT[w_dtype], _ptr(cos_sin),
         _ptr(slots) if store_kv else 0, float(eps), int(bool(store_kv)), _ptr(k_pages), _ptr(v_pages),
         _ptr(order) if order is not None else 0, T,
         _ptr(positions), _ptr(block_tables), block_tables.shape[1], _ptr(out), _ptr(part_m), _ptr(part_l),
         _ptr(part_acc), H, KV, D, bs, float(scale), int(window), part_size, P, _stream())  # fmt: skip


def attn_f32_fresh_supported(dtype, num_heads: int, num_kv_heads: int, head_dim: int, block_size: int, rotary_dim: int, qk_norm: bool) -> bool:
    """Whether `attn_f32_fresh` takes this case: the 32-bit heads that `attn_f32_supported` names, with a per-head norm and rotated whole."""
    return attn_f32_supported(dtype, num_heads, num_kv_heads, head_dim, block_size) and rotary_dim == head_dim and qk_norm


def attn_f32_fresh(qkv, q_weight, k_weight, cos_sin, slots, eps, store_kv, k_pages, v_pages, positions, block_tables, out, num_heads,
                   scale, window, max_context, part_size=None, order=None) -> None:  # fmt: skip
    """`attn_decode_fresh` for 32-bit heads, gains, pages and results: what `qk_norm_rope_store` and then `attn_single_query` do, faster at every size
    measured and as close to 64 bits.  us of this one / of the two, 16 heads on 8 kv heads, by requests x tokens (heads of 128, then of 64; 8, 32 and 40
    heads on 8, 8 on 2 and 16 on 1, steps of several workgroups a compute unit: 1.5 to 16 per cent less in each of 65 sizes):
        1 x 100       4 x 200       32 x 200      64 x 200      4 x 600       8 x 600       16 x 600      4 x 2,000     32 x 2,000    8 x 6,000
        9.4/11.1      13.7/15.1     18.9/20.4     29.0/32.2     13.8/15.2     19.6/21.3     28.9/30.7     21.5/23.6     104/106       77/80
        7.2/8.9       9.6/11.4      11.2/13.1     17.8/20.1     11.5/12.8     13.7/15.5     17.3/19.3     14.2/16.0     55/58         44/46"""
    _check(qkv, "qkv", F32, (None, None, None))
    T, heads, D = qkv.shape
    H = num_heads
    _check(k_pages, "k_pages", F32, (None, None, None, D))
    _, KV, bs, _ = k_pages.shape
    if heads != H + 2 * KV:
        raise KernelError(f"qkv has {heads} heads, expected {H} + 2 x {KV}")
    _check(v_pages, "v_pages", F32, (k_pages.shape[0], KV, D, bs))
    _check(out, "out", F32, (T, H, D))
    _check(positions, "positions", I32, (T,))
    _check(block_tables, "block_tables", I32, (None, None))
    if block_tables.shape[0] < T:
        raise KernelError(f"attention: {T} tokens that are their own rows need as many block tables")
    R = 2 * cos_sin.shape[1] if cos_sin is not None else 0
    if not attn_f32_fresh_supported(F32, H, KV, D, bs, R, q_weight is not None and k_weight is not None):
        raise KernelError(f"attention from fresh projections: unsupported heads {H}/{KV}, head width {D}, "
                          f"rotary width {R}, page size {bs}, or no per-head norm")  # fmt: skip
    _check(cos_sin, "cos_sin", F32, (T, D // 2, 2))
    _check(q_weight, "q_weight", F32, (D,))
    _check(k_weight, "k_weight", F32, (D,))
    if store_kv:
        _check(slots, "slots", I32, (T,))
    if order is not None:
        _check(order, "order", I32, (T,))
    if T == 0:
        return
    if max_context > block_tables.shape[1] * bs:
        raise KernelError("attention: block tables are shorter than the longest context")
    part_size, P, part_m, part_l, part_acc = _partitions(T, H, KV, D, max_context, window, True, part_size, qkv.device)
    call("as_attn_f32_fresh", _ptr(qkv), _ptr(q_weight), _ptr(k_weight), _ptr(cos_sin), _ptr(slots) if store_kv else 0, float(eps),
         int(bool(store_kv)), _ptr(k_pages), _ptr(v_pages), _ptr(order) if order is not None else 0, T, _ptr(positions),
         _ptr(block_tables), block_tables.shape[1], _ptr(out), _ptr(part_m), _ptr(part_l), _ptr(part_acc), H, KV, D, bs, float(scale),
         int(window), part_size, P, _stream())  # fmt: skip


PREFILL_TILE_QUERIES = 64  # queries of one work item of the prefill kernel
PREFILL_MAX_HEAD_DIM = 256  # four stages of 32 keys and values of such heads fill 128 KB of LDS


def attn_prefill_supported(dtype, head_dim: int, block_size: int) -> bool:
    """Whether `attn_prefill` takes this case; if not, the rows go through `attn_single_query`."""
    return dtype == BF16 and head_dim % 32 == 0 and head_dim <= PREFILL_MAX_HEAD_DIM and block_size % 16 == 0


# The prefill attention has two variants: a wave owns 32 queries of a head (two column tiles of 16), four waves two
# heads' 64 queries; or a wave owns 16 and four waves one head's 64, which makes twice the workgroups with half the
# arithmetic each for the same keys and values brought into LDS.  And a step of few work items lasts as long as its
# longest (a portion of 512 tokens behind 15,872 cached ones is 128 workgroups of 256 rounds of 64 keys on a GPU with
# places for 512): every item may come as several workgroups, the items of more rounds than a piece has cut along
# their keys into such pieces and merged by a second kernel (csrc/attention.hip, PrefillSplit).
#
# Which of the two and how many pieces is chosen by a cost in microseconds, fitted to the kernel's times on 96 steps
# (portions of 64 to 4,096 tokens behind 0 to 15,872 cached ones, lone prompts of 128 to 16,384 tokens; 16, 32, 40 and
# 64 heads of 128 on 8 kv heads; 256 compute units; keys and values of 24 layers in turn, so that they come from
# memory): a round costs a workgroup of the first kind 1.5 us when it has a compute unit to itself and 2.2 us when it
# shares one, of the second kind 1.25 and 1.4 us; workgroups beyond the places wait for one, in whole turns when the
# items are equally long and evenly when they are of every length (a lone prompt: one round up to all); the merge
# costs 6 us and what it writes and reads.  What the cost picks is within 1 per cent of the best of the 12 choices on
# average there and 22 per cent at worst (the rule it replaces, cut only while pieces x items fit the places and 16
# queries to a wave only while the workgroups are fewer than the compute units: 2.6 per cent and 38; 512 tokens
# behind 15,872 of Qwen3-8B sizes 213 -> 173 us, of Qwen3-14B sizes 337 -> 268).
PREFILL_QUERY_TILES = None  # 1 or 2 to force a variant (measurements and tests); None: by the cost
PREFILL_PIECES = None  # a number to force that many pieces (1: none; measurements and tests); None: by the cost
PREFILL_PIECE_CHOICES = (1, 2, 3, 4, 6, 8)
PREFILL_MIN_PIECE_ROUNDS = 8  # a piece has at least this many rounds (at 24 rounds in all the merge costs what the cut gains)


def _prefill_units(query_tiles: int, group: int) -> int:
    """Workgroups of four waves that share a tile's queries of one kv head."""
    return -(-(64 // (16 * query_tiles)) * group // 4)


def _prefill_cost(num_tiles: int, H: int, KV: int, D: int, rounds: int, mean_rounds: float, query_tiles: int,
                  pieces: int, tokens: int) -> float:  # fmt: skip
    """Microseconds, roughly, of a prompt step's attention: `num_tiles` tiles of 64 queries, the longest item of
    `rounds` rounds of 64 keys, the items of `mean_rounds` on average."""
    group, wide = H // KV, D / 128
    alone, shared = ((1.5, 2.2) if query_tiles == 2 else (1.25, 1.4))
    per_cu = 2 if D <= 128 else 1  # the rings of wider heads leave room for one workgroup
    if per_cu == 1:
        shared = alone
    places = per_cu * compute_units()
    workgroups = num_tiles * KV * _prefill_units(query_tiles, group) * pieces
    piece_rounds = -(-rounds // pieces)
    if workgroups <= compute_units():
        cost = piece_rounds * alone
    elif workgroups <= places:
        cost = piece_rounds * shared
    else:
        work = num_tiles * KV * (64 // (16 * query_tiles)) * group / 4 * pieces  # in full workgroups
        spread = min(1.0, max(0.0, 2.0 * (1.0 - mean_rounds / rounds)))  # 0: all items as long as the longest; 1: of every length
        evenly = max(piece_rounds * shared, (work * mean_rounds / pieces / places + 0.5 * piece_rounds) * shared)
        in_turns = -(-workgroups // places) * piece_rounds * shared
        cost = spread * evenly + (1.0 - spread) * in_turns
    cost *= wide
    if pieces > 1:
        cost += 6.0 + tokens * H * pieces * D * 8 / 2e6  # partial results written and read at 2 TB/s
    return cost + 6.0


def _prefill_plan(num_tiles: int, H: int, KV: int, D: int, max_context: int, window: int = 0, query_tiles=None,
                  tile_keys: int = 0, keep_first: int = 0) -> tuple:  # fmt: skip
    """(query tiles of a wave, pieces, rounds of a piece) for a prompt step; pieces 1 (and 0 rounds): nothing is cut.
    tile_keys: the keys that the tiles' last queries see, added up (0: not known; the tiles are then taken to be one
    request's last ones).  Every layer of a step asks the same question: the answers are kept."""
    if query_tiles is None:
        query_tiles = PREFILL_QUERY_TILES
    return _prefill_plan_of(num_tiles, H, KV, D, max_context, window, query_tiles, tile_keys, PREFILL_PIECES, compute_units(), keep_first)


def _prefill_rounds(num_tiles, max_context, window, tile_keys, keep_first=0) -> tuple:
    """Rounds of 64 keys of the longest item, and of the items on average."""
    span = min(max_context, window + 64 + keep_first) if window > 0 else max_context  # the keys that the longest item walks
    rounds = max(1, -(-span // 64))
    if tile_keys > 0:
        return rounds, min(rounds, max(1.0, tile_keys / num_tiles / 64))
    return rounds, max(rounds - num_tiles / 2, rounds / 2)


@functools.lru_cache(maxsize=1024)
def _prefill_plan_of(num_tiles, H, KV, D, max_context, window, query_tiles, tile_keys, forced_pieces, units, keep_first=0) -> tuple:
    rounds, mean_rounds = _prefill_rounds(num_tiles, max_context, window, tile_keys, keep_first)
    kinds = (2, 1) if query_tiles is None else (int(query_tiles),)
    if forced_pieces is not None:
        cuts = (max(1, min(int(forced_pieces), rounds // 2)),)
    else:
        cuts = tuple(c for c in PREFILL_PIECE_CHOICES if c == 1 or rounds // c >= PREFILL_MIN_PIECE_ROUNDS)
    tokens = 64 * num_tiles
    kind, pieces = min(((k, c) for k in kinds for c in cuts),
                       key=lambda kc: _prefill_cost(num_tiles, H, KV, D, rounds, mean_rounds, kc[0], kc[1], tokens))  # fmt: skip
    return (kind, pieces, -(-rounds // pieces)) if pieces > 1 else (kind, 1, 0)


def attn_prefill(q, k_pages, v_pages, tiles, block_tables, out, scale, window, max_context, query_tiles=None,
                 tile_keys: int = 0, keep_first=0, softcap=0.0, sink=False, chunk=0) -> None:  # fmt: skip
    """Causal attention of prompt portions over the paged cache, bfloat16, on the matrix cores.

    tiles [Nt, 4] int32: (first flat token, count <= 64, block-table row, position of the first
    token) of up to 64 consecutive tokens of one request; the keys of these tokens are already in
    the pages.  max_context: host bound on the last position + 1 of any tile.
    query_tiles: column tiles of 16 queries that a wave owns, 2 or 1; None: chosen here.
    tile_keys: the sum over the tiles of (position of the first token + count), if the caller knows it: how the
    work is cut is chosen better with it (speed only).
    window, keep_first, softcap, sink, chunk: as for `attn_single_query`."""
    _check(q, "q", BF16, (None, None, None))
    T, H, D = q.shape
    sight = _sight(window, keep_first, chunk, softcap, sink, q, out)
    _check(k_pages, "k_pages", BF16, (None, None, None, D))
    _, KV, bs, _ = k_pages.shape
    _check(v_pages, "v_pages", BF16, (k_pages.shape[0], KV, D, bs))
    _check(tiles, "tiles", I32, (None, 4))
    _check(block_tables, "block_tables", I32, (None, None))
    if tiles.shape[0] == 0:
        return
    if H % KV or not attn_prefill_supported(q.dtype, D, bs):
        raise KernelError(f"prefill attention: unsupported heads {H}/{KV}, head width {D} or page size {bs}")
    if max_context > block_tables.shape[1] * bs:
        raise KernelError("attention: block tables are shorter than the longest context")
    query_tiles, pieces, piece_rounds = _prefill_plan(tiles.shape[0], H, KV, D, max_context, window or chunk, query_tiles, tile_keys, sight[1])
    cut = part_ml = part_acc = None
    if pieces > 1:
        cut = torch.empty(tiles.shape[0] * KV * _prefill_units(query_tiles, H // KV), dtype=I32, device=q.device)
        part_ml = torch.empty((T, H, pieces, 2), dtype=F32, device=q.device)
        part_acc = torch.empty((T, H, pieces, D), dtype=F32, device=q.device)
    call("as_attn_prefill_mfma", _ptr(q), _ptr(k_pages), _ptr(v_pages), _ptr(tiles), tiles.shape[0],
         _ptr(block_tables), block_tables.shape[1], _ptr(out), H, KV, D, bs, float(scale), *sight,
         int(query_tiles), pieces, piece_rounds, _ptr(cut), _ptr(part_ml), _ptr(part_acc), _stream())  # fmt: skip


def attn_mixed_supported(dtype, H: int, KV: int, D: int, block_size: int) -> bool:
    """Whether `attn_mixed` takes these heads and pages (with a window at most: no kept tokens, caps, sinks or chunks)."""
    return dtype == BF16 and D in (64, 128) and block_size == 16 and H % KV == 0 and H // KV <= 16


# Both kinds of work in one launch, single queries first.  How the portions' items and the singles' contexts are cut is chosen together, by a cost in
# microseconds fitted to 22,000 times of 614 steps (1 to 128 single queries of up to 8,000 keys beside portions of 9 to 4,000 tokens behind up to
# 14,000; 16 to 64 heads of 128 on 8 kv heads, 1, 2 and 4 kv heads, heads of 64; 256 compute units): a round of 64 keys is 1.4 us of a workgroup
# of the portions' first kind and 2.05 of the second, with heads of 64 a tenth more; a single query's partition 5 us and 12 ns a key (contexts:
# three fifths of the longest on average).  Workgroups that all have a place (two to a compute unit, 3.2 with heads of 64) last as long as the longest
# of them.  More of them last for all the work divided by the places and for a quarter of a piece at the end, and halfway from there to whole
# turns as far as the items are equally long.  Merges cost 6 us and 2 TB/s for what pieces leave, 4.1 us, 0.3 a partition and 1.5 TB/s for what singles
# leave.  What it picks takes 1.7 per cent more than the best form on average and 24 at worst, on 160 other steps 1.9 and never more than two
# launches; two steps of the 614 take 2 to 4 per cent more.  (Without places and turns, pieces by 10 us and 5 TB/s: 4.2 per cent, 40 at worst, and 31
# steps, of long portions beside few or short contexts, took 2 to 27 per cent more than two launches; one of 1,274 tokens behind 4,530 beside one query, 40 heads,
# two launches 201, then 237, now 193.)
# One layer, us, two launches / this (best of all forms): Qwen3-8B sizes, 32 of 100 to 2,048 keys beside 480 tokens behind 7,001 145 / 126 (122), 8 of 2,048
# beside 504 34 / 27.8 (27.8), 8 of 500 to 8,192 beside 504 60 / 42 (40), 96 of 200 to 600 beside 2,000 100 / 95 (91), 20 of 1,000 to 3,000 beside four of 120 behind
# 6,000 163 / 126 (117); 40 heads, 128 of 32 to 400 beside 384 behind 2,000 74 / 76 (67); 16 heads, 4 of 300 to 900 beside 37 15.0 / 12.0 (11.1).
@functools.lru_cache(maxsize=1024)
def _mixed_plan(num_tiles: int, H: int, KV: int, D: int, tile_context: int, tile_keys: int, singles: int, single_context: int,
                window: int, units: int, query_tiles=None, forced_pieces=None) -> tuple:  # fmt: skip
    """(query tiles of a wave, pieces, rounds of a piece, keys of a single query's partition) for a step of both kinds; query_tiles,
    forced_pieces: numbers to force, as PREFILL_QUERY_TILES and PREFILL_PIECES."""
    rounds, mean_rounds = _prefill_rounds(num_tiles, tile_context, window, tile_keys)
    span = _seen_keys(single_context, window, 0, True)
    places, whole, groups = (2.0 if D > 64 else 3.2) * units, _up32(span), singles * KV
    # What depends on the singles' cut alone, and on the portions' alone, is worked out once: a step's lengths are new ones, so that a plan is made in each.
    ways = []
    for part in (whole, *[n for n in MFMA_PARTITIONS if n < whole]):
        parts = -(-span // part)
        merge = MERGE_LAUNCH + 0.3 * parts + singles * H * parts * D * 8 / 1.5e6 if parts > 1 else 0.0
        ways.append((part, groups * parts, groups * (5.0 * parts + 0.012 * 0.6 * span), 2.75 + 0.0125 * min(part, span), merge))
    turning = 0.5 * (1.0 - min(1.0, max(0.0, 2.0 * (1.0 - mean_rounds / rounds))))  # 0: items of every length
    kinds = ((1, 1.4), (2, 2.05)) if D > 64 else ((1, 1.54), (2, 2.255))
    if query_tiles is not None:
        kinds = (kinds[int(query_tiles) - 1],)
    if forced_pieces is not None:
        cuts = (max(1, min(int(forced_pieces), rounds // 2)),)
    else:
        cuts = [c for c in PREFILL_PIECE_CHOICES if c == 1 or rounds // c >= PREFILL_MIN_PIECE_ROUNDS]
    best = None
    for kind, round_time in kinds:
        workgroups = num_tiles * KV * _prefill_units(kind, H // KV)
        work = workgroups * mean_rounds * round_time
        for pieces in cuts:
            piece = -(-rounds // pieces) * round_time
            turns = -(-workgroups * pieces // places) * piece
            merge = 6.0 + 64 * num_tiles * H * pieces * D * 8 / 2e6 if pieces > 1 else 0.0
            for part, single_groups, single_work, single, single_merge in ways:
                cost = piece if piece > single else single
                if workgroups * pieces + single_groups > places:
                    evenly = (work + single_work) / places + 0.25 * piece
                    busy = evenly + turning * (turns - evenly)
                    cost = busy if busy > cost else cost
                cost += merge + single_merge
                if best is None or cost < best[0]:
                    best = (cost, kind, pieces, part)
    _, kind, pieces, part = best
    return kind, pieces, -(-rounds // pieces) if pieces > 1 else 0, part


def attn_mixed(q, k_pages, v_pages, items, tiles, positions, tok_row, block_tables, out, scale, window, max_tile, max_single,
               tile_keys: int = 0) -> None:  # fmt: skip
    """`attn_single_query` of the tokens `items` and `attn_prefill` of the portions `tiles` in one launch, for steps that
    `attn_mixed_supported` takes: arguments as there; max_tile, max_single: host bounds on the last position + 1 of a tile and on
    positions[items] + 1."""
    _check(q, "q", BF16, (None, None, None))
    T, H, D = q.shape
    _check(out, "out", BF16, (T, H, D))
    _check(k_pages, "k_pages", BF16, (None, None, None, D))
    _, KV, bs, _ = k_pages.shape
    _check(v_pages, "v_pages", BF16, (k_pages.shape[0], KV, D, bs))
    _check(items, "items", I32, (None,))
    _check(tiles, "tiles", I32, (None, 4))
    _check(positions, "positions", I32, (T,))
    _check(tok_row, "tok_row", I32, (T,))
    _check(block_tables, "block_tables", I32, (None, None))
    N, tile_count, dev = items.shape[0], tiles.shape[0], q.device
    if N == 0 or tile_count == 0 or not attn_mixed_supported(q.dtype, H, KV, D, bs):
        raise KernelError(f"mixed attention: {N} single queries, {tile_count} tiles, heads {H}/{KV} of {D}, pages of {bs}")
    if max(max_tile, max_single) > block_tables.shape[1] * bs:
        raise KernelError("attention: block tables are shorter than the longest context")
    kind, pieces, piece_rounds, part = _mixed_plan(tile_count, H, KV, D, max_tile, tile_keys, N, max_single, window, compute_units(),
                                                   PREFILL_QUERY_TILES, PREFILL_PIECES)  # fmt: skip
    part_size, P, part_m, part_l, part_acc = _partitions(N, H, KV, D, max_single, window, True, part, dev)
    cut = piece_ml = piece_acc = None
    if pieces > 1:
        cut = torch.empty(tile_count * KV * _prefill_units(kind, H // KV), dtype=I32, device=dev)
        piece_ml = torch.empty((T, H, pieces, 2), dtype=F32, device=dev)
        piece_acc = torch.empty((T, H, pieces, D), dtype=F32, device=dev)
    call("as_attn_mixed_mfma", _ptr(q), _ptr(k_pages), _ptr(v_pages), _ptr(tiles), tile_count, _ptr(items), N, _ptr(positions),
         _ptr(tok_row), _ptr(block_tables), block_tables.shape[1], _ptr(out), H, KV, D, bs, float(scale), window, int(kind),
         pieces, piece_rounds, _ptr(cut), _ptr(piece_ml), _ptr(piece_acc), _ptr(part_m), _ptr(part_l), _ptr(part_acc),
         part_size, P, _stream())  # fmt: skip


SKINNY_MAX_ROWS = 16  # up to here the bf16 product streams the weights through our own kernel
# 17 to 32 rows: the persistent kernel keeps two row tiles in registers up to this K ...
SKINNY_TWO_MAX_ROWS, SKINNY_TWO_MAX_K = 32, 4096
# ... and pays while the activations, which EVERY workgroup reads whole, stay a fraction of the
# weights' bytes: at 32 rows of 4096 over 256 workgroups (67 MB) the library's product is faster,
# with rows of 1024 (17 MB) this one is, by the two kernels it saves beside.
SKINNY_TWO_MAX_ACT_BYTES = 36 << 20


def _workgroups() -> int:
    """Persistent kernels run one workgroup per compute unit."""
    return compute_units()



def _few_rows(rows: int, k: int, n: int, max_k=None, w=None) -> bool:
    """Whether a product of `rows` rows of width `k` with `n` output columns goes through the
    few-rows kernels of this package.  w: the weights, if known: with a copy in wave order, 17 to 32
    rows are left to the tile products (and the library), which are then the faster ones, also for narrow
    rows (Qwen3-0.6B sizes, batch 32: 12,430 -> 12,580 to 12,750 tokens/s), and so are 9 to 16 rows of a
    model that is wide enough (`_tile_preferred`; Qwen3-8B sizes, batch 16: 3,497 -> 3,594, batch 9: 2,045
    -> 2,106; at 8 rows and fewer the few-rows kernels win: 2,129 against 2,019)."""
    if rows <= 0 or k % 8:
        return False
    if w is not None and _tile_preferred(rows, k, n, w):
        return False
    if rows <= SKINNY_MAX_ROWS:
        return max_k is None or k <= max_k
    strips = min(-(-n // 16), _workgroups())
    return (rows <= SKINNY_TWO_MAX_ROWS and k <= SKINNY_TWO_MAX_K
            and strips * rows * k * 2 <= SKINNY_TWO_MAX_ACT_BYTES)  # fmt: skip


def few_rows_product(a, w) -> bool:
    """Whether `gemm` of these bf16 matrices with bf16 results goes through the few-rows kernels."""
    return a.dtype == BF16 and _few_rows(a.shape[0], a.shape[1], _rows(w).shape[0], w=w)


def gemm(a, w, out, choices=None) -> None:
    """out[M, N] = a[M, K] @ w[N, K]^T.  fp32: own kernel (32-bit operands and sums; above 256 columns every float as three bf16
    parts, six products of parts for one, with an error no larger than the fp32 instruction's).  bf16: own kernel for few
    rows, the library's matrix product otherwise; `out` may be bf16 or (few rows) fp32.
    w: a tensor, or a `Streamed`.  choices: the `ProductChoices` that says which of the library's kernels
    runs (a model's own; None: the one the process shares)."""
    _check(a, "a", (F32, BF16), (None, None))
    M, K = a.shape
    rows = _rows(w)
    _check(rows, "w", a.dtype, (None, K))
    N = rows.shape[0]
    _check(out, "out", None, (M, N))
    if M == 0:
        return
    if a.dtype == F32:
        _check(out, "out", F32)
        call("as_gemm_f32", _ptr(a), _ptr(rows), _ptr(out), M, N, K, 0, _stream())
        return
    if out.dtype not in (BF16, F32):
        raise KernelError(f"gemm: unsupported output dtype {out.dtype}")
    if _few_rows(M, K, N, w=w if out.dtype == BF16 else None):  # fp32 results (the head): no tile product to prefer
        call("as_gemm_bf16_skinny", _ptr(a), _ptr(rows), _wave_ptr(w), _ptr(out), _DT[out.dtype], M, N, K, 0, _stream())
        return
    strips = _wide_tile_strips(M, N, K) if out.dtype == F32 and _wave_ptr(w) else 0
    if strips and M <= WIDE_TILE_ALWAYS_ROWS and a.data_ptr() % 16 == 0:
        call("as_gemm_bf16_tile", _ptr(a), _ptr(rows), _wave_ptr(w), _ptr(out), 0, _DT[F32], M, N, K, 0, 0, strips, _stream())
    else:
        (choices or SHARED).gemm(a, w, out, M, N, K)


# ---- the library's product, called directly -------------------------------------------------
#
# hipBLASLt through `csrc/blas.hip` instead of torch.mm: the same kernels for two thirds of the
# time on the host.  For the row counts that a `ProductChoices` is told to tune (decode steps of 17
# and more requests are padded to a few row counts, which the capture of such a step names, and are
# replayed thousands of times) the library's first candidate is often not its fastest on this GPU, so
# the first calls of such a shape try the candidates in turn, each on the weights of the layer that
# happens to call (cold, as every decode step meets them), timed by events in place; when every
# candidate has run LIBRARY_TRIALS_EACH times (the first run of a kernel is slow), or a capture
# begins, the fastest stays.  The same is done for the token budget of a step and for lengths of
# prompts that a warm-up runs, and a product of any other row count above 64 takes the kernel that
# the nearest tuned row count above it settled on: at 128 rows of Qwen3-8B sizes the library's first
# candidates take 168 us a layer, the fastest of the first sixteen 132 us.
LIBRARY_WORKSPACE_BYTES = 64 << 20
LIBRARY_DECODE_ROWS = 64  # row counts up to here are decode steps' (padded to 32, 48 and 64)
LIBRARY_TRIALS_EACH = 4
SETTLE_EACH = 2  # runs of every candidate behind the fills that let the host get ahead, before a capture
_workspace = {}  # device index -> the library's scratch memory, one for the process (its calls follow one another)

# Beside the library's candidates a trial may time this package's plain tile product (9 to 128 rows, K in
# chunks of 256, bf16 out, weights with a copy in wave order) with tiles of 2 and of 4 strips: for qkv
# of Qwen3-8B sizes it takes 12.7 / 14.8 / 16.3 us at 32 / 48 / 64 rows against the library's best 14.7 /
# 17.3 / 17.6; for the 4,096 columns of o the library wins at 32 to 64 rows.  With 32-bit results (the head) the tile
# product of 65 to 96 rows is such a candidate too (`_wide_tile_strips`).  Such a candidate's number is OWN_CANDIDATE + its strips.
# Above 128 rows the tile of the large products (`_wide_plan`) is one, WIDE_CANDIDATE, where it may win: 4,096 columns of K = 1,024, 512 rows
# 10.7 us against the library's best 11.8, 1,024 rows 11.4 against 14.4; 4,096 of 4,096, 1,024 rows 36 against 39; 6,144 of 2,560, 2,048 rows
# 52 against 55; lost by a tenth and more where there are few outputs and a long K.
OWN_CANDIDATE, WIDE_CANDIDATE = 1000, 2000
WIDE_PLAIN_MIN_OUTPUTS = 1024


def _library_workspace(device):
    """The library's scratch memory on `device`; None inside a capture that finds none yet (nothing is
    allocated for good there)."""
    index = device.index if device.index is not None else torch.cuda.current_device()
    space = _workspace.get(index)
    if space is None and not torch.cuda.is_current_stream_capturing():
        space = _workspace[index] = torch.empty(LIBRARY_WORKSPACE_BYTES, dtype=torch.uint8, device=device)
    return space


def _torch_gemm(a, w, out) -> None:
    watch.spoiled = True  # no call of an entry point
    w = _rows(w)
    if out.dtype == BF16:
        torch.mm(a, w.t(), out=out)
    else:
        out.copy_(torch.mm(a, w.t()))


def _own_candidates(M, N, K, dtype, w) -> list:
    """w: the weights, to see whether they have a copy in wave order; None: taken for granted."""
    if dtype == F32 and (w is None or _wave_ptr(w)):
        strips = _wide_tile_strips(M, N, K)
        return [OWN_CANDIDATE + strips] if strips else []
    if dtype == BF16 and _wide_sizes(M, N, N, K):
        return [WIDE_CANDIDATE] if N >= WIDE_PLAIN_MIN_OUTPUTS and _wide_plan(M, N, K, WIDE_PLAIN)[0] <= 1.1 * _library_us(M, N, K) else []
    if dtype != BF16 or not _tile_rows(M, K, BF16, TILE_SPLIT_MAX_ROWS) or N % 16:
        return []
    if w is not None and not _wave_ptr(w):
        return []
    return [OWN_CANDIDATE + 2, OWN_CANDIDATE + 4]


def _own_call_possible(a, w, out, candidate) -> bool:
    """Whether this package's product `candidate` can run on these matrices (it was chosen for their sizes, on others)."""
    if candidate >= WIDE_CANDIDATE:
        return _wide_takes(a, w, out.shape[1], out.shape[1]) and out.data_ptr() % 16 == 0
    return bool(_wave_ptr(w)) and not (out.dtype == F32 and a.data_ptr() % 16)


def _library_call(a, w, out, M, N, K, candidate) -> None:
    if candidate >= WIDE_CANDIDATE:
        if not _own_call_possible(a, w, out, candidate):
            raise KernelError("the large tiles were chosen for matrices that start on 16 bytes")
        call("as_gemm_bf16_wide", _ptr(a), _ptr(_rows(w)), _ptr(out), M, N, K, WIDE_PLAIN, 1, _wide_plan(M, N, K, WIDE_PLAIN)[1], _stream())
        return
    if candidate >= OWN_CANDIDATE:
        if not _wave_ptr(w) or (out.dtype == F32 and a.data_ptr() % 16):
            raise KernelError("the tile product was chosen for weights with a copy in wave order and rows that start on 16 bytes")
        call("as_gemm_bf16_tile", _ptr(a), _ptr(_rows(w)), _wave_ptr(w), _ptr(out), 0, _DT[out.dtype], M, N, K, 0, 0,
             candidate - OWN_CANDIDATE, _stream())  # fmt: skip
        return
    call("as_blas_gemm", _ptr(a), _ptr(_rows(w)), _ptr(out), _DT[out.dtype], M, N, K, candidate,
         _ptr(_library_workspace(a.device)), LIBRARY_WORKSPACE_BYTES, _stream())  # fmt: skip


def prepare_library_adoption() -> bool:
    """Pays the library's one-time cost of finding a kernel by its number (a third of a second) now, not
    at the first prompt of a length that was not tuned.  False while no shape has been planned."""
    return bool(entry("as_blas_prepare_adoption")())


class ProductChoices:
    """Which kernel runs for each shape of the matrix products that the few-rows kernels leave over: one
    of the library's candidates or one of this package's tile products, settled by timed trials for the
    row counts it is told to tune, or always the library's first (`fixed`).  A model owns one (its parts
    hand it to `gemm`), so what is chosen on one model's weights, which row counts are tuned and whether
    choices are fixed belong to that model's engine or tool and to no other in the process; calls that
    name none share `SHARED`."""

    def __init__(self, fixed: bool = False):
        self.fixed = bool(fixed)
        self.choice = {}  # (rows, columns, width, output dtype) -> candidate
        self.library = {}  # the same key -> the library's fastest candidate of the trial, where a product of this package won it
        self.trials = {}  # the same key -> a trial under way
        self.tuned_rows = {32, 48, 64}

    def fix(self, fixed: bool = True) -> None:
        """fixed: every shape not settled yet takes the library's first candidate (what torch.mm runs)
        instead of timing the candidates, so that bfloat16 results are the same from process to process.
        Choices already made stay (they were made under the setting of their time)."""
        self.fixed = bool(fixed)
        if fixed:
            self.trials.clear()

    def chosen(self) -> dict:
        """(rows, columns, width, output dtype) -> the candidate that runs, for every shape settled so far
        (-1: torch's own call; OWN_CANDIDATE + strips, WIDE_CANDIDATE: this package's tile products); enough to reproduce a
        run's products."""
        return dict(self.choice)

    def tune_rows(self, rows: int) -> None:
        """Also try the candidates for products of this many rows: a row count that comes again and
        again, like the token budget of the steps that carry a portion of a prompt."""
        self.tuned_rows.add(int(rows))

    def wants_trial(self, M, N, K) -> bool:
        """Whether the kernels of this product with bf16 results are still to be tried (or are being tried) by calls like this one.  What a
        rule gives to a kernel beside the trials (a gated product, sums in parts) waits until they have been, though this row count has no use
        for them then: the row counts that follow it may fall on the library's side of the rule (5,120 outputs of K = 17,408, 800 rows, whole,
        under 1,024, cut: 234 us with the library's first kernel, 177 with the one that the trial at 1,024 rows names; 2,560 of 9,728, 900
        rows: 77 and 68; a prompt of 800 tokens through 6 layers of Qwen3-14B sizes 5.04 and 4.38 ms)."""
        return (M in self.tuned_rows and not self.fixed and (M, N, K, BF16) not in self.choice
                and not torch.cuda.is_current_stream_capturing())  # fmt: skip

    def trials_pending(self) -> bool:
        """Whether some shape is still trying candidates (a warm-up may then run once more)."""
        return bool(self.trials)

    def gemm(self, a, w, out, M, N, K) -> None:
        key = (M, N, K, out.dtype)
        choice = self.choice.get(key)
        if choice is None:
            capturing = torch.cuda.is_current_stream_capturing()
            if _library_workspace(a.device) is None:
                return _torch_gemm(a, w, out)  # inside a capture, before any call outside one: torch's own call this once
            trial = self.trials.get(key)
            if trial is None:
                count = entry("as_blas_plan")(M, N, K, _DT[out.dtype], LIBRARY_WORKSPACE_BYTES)
                if count == 0:
                    choice = self.choice[key] = -1  # the library offers nothing for this shape through this door
                elif self.fixed or (count == 1 and not _own_candidates(M, N, K, out.dtype, w)):
                    choice = self.choice[key] = 0  # the library's first candidate, which is what torch.mm runs
                elif _plain_tile_strips(M, N, K, out.dtype) and _own_candidates(M, N, K, out.dtype, w):
                    choice = self.choice[key] = OWN_CANDIDATE + _plain_tile_strips(M, N, K, out.dtype)
                elif M not in self.tuned_rows:
                    choice = self._choice_of_tuned_rows(M, N, K, out.dtype)  # a prompt of any length: what its bucket settled on
                    if choice is None:
                        choice = 0  # nothing settled yet: the first candidate for now, asked again at the next call
                    else:
                        self.choice[key] = choice
                else:
                    ids = list(range(count)) + _own_candidates(M, N, K, out.dtype, w)
                    trial = self.trials[key] = {"count": len(ids), "ids": ids, "runs": [], "weights": []}
            if trial is not None:
                if not capturing and not _tried_enough(trial):
                    trial["last"] = (a, w, out)
                    if not any(w is met for met in trial["weights"]):
                        trial["weights"].append(w)
                    _trial_run(trial, a, w, out, M, N, K)
                    return
                choice = self._end_trial(key, self.trials.pop(key))
        if choice < 0:
            return _torch_gemm(a, w, out)
        if choice >= OWN_CANDIDATE and not _own_call_possible(a, w, out, choice):
            # chosen on weights that had a copy in wave order, or on aligned rows; these have none, or are not
            choice = self._library_choice(key)
        _library_call(a, w, out, M, N, K, choice)

    def _end_trial(self, key, trial) -> int:
        choice = self.choice[key] = _fastest_of(trial)
        if choice >= OWN_CANDIDATE:
            self.library[key] = _fastest_of(trial, OWN_CANDIDATE)
        return choice

    def _library_choice(self, key) -> int:
        """The library's candidate for a settled shape on whose matrices this package's product, which was chosen, cannot run: the
        fastest of the shape's own trial, or of the row count's that this one follows; its first where no trial said."""
        place = self.library.get(key)
        if place is None and not self.fixed and key[0] not in self.tuned_rows:
            place = self._choice_of_tuned_rows(*key, own=False)
            if place is not None:
                self.library[key] = place
        return place or 0

    def _choice_of_tuned_rows(self, M, N, K, dtype, own: bool = True):
        """For a product of a row count that is not tuned itself: the kernel that the nearest tuned row
        count above it (of more than 64 rows: a prompt's, not a decode step's) settled on for the same
        weights, as a candidate of this shape; None while that one has not settled, or there is none.
        Where that is a product of this package which is no candidate here (or `own` is not asked for): the
        fastest of the library's there (4,096 columns of K = 4,096, 1,300 rows under 1,536, where the large tile had won: 47.7 us with
        the library's first, 46.4 with that one)."""
        above = [rows for rows in self.tuned_rows if rows >= M and rows > LIBRARY_DECODE_ROWS]
        if not above:
            return None
        tuned = min(above)
        settled = self.choice.get((tuned, N, K, dtype))
        if settled is None:
            return None
        if settled < 0:
            return 0
        if settled >= OWN_CANDIDATE:  # this package's tile kernel: for this row count too if it takes it
            if own and settled in _own_candidates(M, N, K, dtype, None):
                return settled
            settled = self.library.get((tuned, N, K, dtype), 0)
        index = entry("as_blas_candidate_index")(tuned, N, K, _DT[dtype], LIBRARY_WORKSPACE_BYTES, settled)
        place = entry("as_blas_adopt")(M, N, K, _DT[dtype], LIBRARY_WORKSPACE_BYTES, index)
        return place if place >= 0 else 0

    @torch.inference_mode()
    def settle(self) -> None:
        """Ends every trial that is under way.  Called before a capture begins, so that the captured
        launches are the ones later replays should make.  In a pass the host is often the slower one, and a run's
        time then is the host's between its two events (a kernel of 9 us came out at 10 to 28).  So each candidate runs
        again here, SETTLE_EACH times behind fills of the library's scratch memory that let the host get
        ahead and, between the runs, push the weights out of the caches: on the rows of the last call and in turn all
        the weights that the trial has met.  Large products, which the host does not hold up, run what is left of their runs."""
        for key in list(self.trials):
            trial = self.trials.pop(key)
            a, _, out = trial["last"]
            small = key[0] <= LIBRARY_DECODE_ROWS
            runs = SETTLE_EACH * trial["count"] if small else LIBRARY_TRIALS_EACH * trial["count"] - len(trial["runs"])
            if small:
                trial["ahead"], space = len(trial["runs"]), _library_workspace(a.device)
                for _ in range(runs):
                    space.zero_()
            for _ in range(runs):
                if small:
                    space[: LIBRARY_WORKSPACE_BYTES // 4].zero_()
                _trial_run(trial, a, trial["weights"][len(trial["runs"]) % len(trial["weights"])], out, *key[:3])
            torch.cuda.current_stream().synchronize()
            self._end_trial(key, trial)


SHARED = ProductChoices()  # for products whose caller names no choices of its own (tools, tests, toy parts)


def _tried_enough(trial) -> bool:
    return len(trial["runs"]) >= LIBRARY_TRIALS_EACH * trial["count"]


def _trial_run(trial, a, w, out, M, N, K) -> None:
    """Computes the product with the candidate whose turn it is, between two events."""
    watch.spoiled = True  # the next call tries another candidate
    candidate = trial["ids"][len(trial["runs"]) % trial["count"]]
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    try:
        _library_call(a, w, out, M, N, K, candidate)
    except KernelError:  # a candidate that does not run; the first one does
        trial["runs"].append((candidate, None, None))
        _library_call(a, w, out, M, N, K, 0)
        return
    end.record()
    trial["runs"].append((candidate, start, end))


def _fastest_of(trial, below=None) -> int:
    """The candidate (of a number under `below`, if given) whose shortest run took least, among the runs that were timed and have finished: those with the host ahead
    (`settle`) where every candidate has one, else all but each candidate's first (which loads the kernel); 0 if none.  (The host
    between a run's two events lengthens it; the caches, which could shorten it, do not hold its weights: a pass comes back to
    them after all others.  On averages qkv of 16 rows at Qwen3-4B sizes went to 12.5 us instead of 9.3 in one process of three.)"""
    times, ahead = {}, {}
    for n, (candidate, start, end) in enumerate(trial["runs"]):
        if start is not None and (below is None or candidate < below) and end.query():
            times.setdefault(candidate, []).append(start.elapsed_time(end))
            if n >= trial.get("ahead", n + 1):
                ahead.setdefault(candidate, []).append(times[candidate][-1])
    if ahead.keys() != times.keys():
        ahead = {candidate: took[1:] or took for candidate, took in times.items()}
    return min(ahead, key=lambda candidate: min(ahead[candidate]), default=0)


# ---- 17 to 128 rows: tiles of weight rows with the activations staged in LDS --------------------
# (above 64 rows in row tiles of 96 and 128.  At 128 rows the library needs 42 us for Qwen3-8B's down
# projection and 21 for o, the split product 24 on average; the gated product of 96 and 128 rows lost to
# the library's with the activation after it while it read the weights from rows, 51 and 61 us against
# 48 and 56, and wins by a little since it reads them in wave order: batch 96 9,507 -> 9,587 tokens/s)
TILE_MAX_ROWS = 128
TILE_SPLIT_MAX_ROWS = 128
TILE_CHUNK = 256  # K comes in chunks of this many


TILE_MIN_ROWS = 9  # up to 8 rows the few-rows kernels are the faster ones in any case (one row tile of 16, half of it padding)
# ... and at 9 to 16 rows while the model is narrow: with their residual sum and norm folded in they save two
# launches a layer, which a small model's step is made of (decode at batch 16, tile products from 9 rows against
# from 17: Qwen3-0.6B sizes 8,391 against 9,082 tokens/s, -1.7B 7,030 against 7,311, -4B 4,697 against 4,499,
# -8B 3,594 against 3,497, -14B 2,311 against 2,069)
TILE_FROM_9_MIN_WIDTH = 2560


def _tile_rows(rows: int, k: int, dtype, most: int = TILE_MAX_ROWS) -> bool:
    return dtype == BF16 and TILE_MIN_ROWS <= rows <= most and k % TILE_CHUNK == 0


def _tile_preferred(rows: int, k: int, n: int, w) -> bool:
    """Whether a product of 9 to 32 rows that the few-rows kernels could take is left to the tile products
    (and the library with them as candidates): weights with a copy in wave order, a K in whole chunks, and
    above 16 rows or a model wide enough (the narrower of k and n is the stream's width in all four
    products of a layer)."""
    return bool(_wave_ptr(w)) and _tile_rows(rows, k, BF16) and (rows > SKINNY_MAX_ROWS or min(k, n) >= TILE_FROM_9_MIN_WIDTH)


WIDE_TILE_MAX_ROWS = 96
WIDE_TILE_ALWAYS_ROWS = 64  # above: one more candidate beside the library's in the timed trials


def _wide_tile_strips(rows: int, n: int, k: int) -> int:
    """Strips of 16 weight rows per workgroup of the tile kernel for a product with 32-bit results and outputs enough to
    fill the GPU several times (the head), 0 where only the library's product runs: 17 to 96 rows and K in whole chunks.
    151,936 outputs, the tile kernel against the library's best of 16 and its first (which a step of an untuned row count takes):
    K            33 rows            64 rows            80 rows            96 rows
    1,024     60   80   80       69   79   85       89   82   87       90   86   88
    2,048    120  141  156      128  153  159      142  156  158      144  161  171
    2,560    143  156  175      160  167  184      177  170  176      182  180  196
    4,096    231  240  255      243  252  269      258  266  273      269  276  278
    5,120    270  294  294      294  293  313      321  305  317      329  328  331
    so up to 64 rows it runs, above them it is tried; at 128 rows and K = 4,096 the library's best takes 287 against 297.
    Few rows want narrow tiles (17 rows, K = 2,048: 2 strips 99 us, 4 strips 114; 64 rows 144, 134 and 8 strips 128)."""
    if not SKINNY_MAX_ROWS < rows <= WIDE_TILE_MAX_ROWS or k % TILE_CHUNK or n % 16 or n * k * 2 > 0xF0000000:
        return 0
    strips = 2 if rows <= 24 else 4 if rows <= 32 or (k <= 1024 and rows <= 64) else 8
    return strips if n >= 16 * strips * compute_units() else 0


PLAIN_TILE_MAX_ROWS = 64


def _plain_tile_strips(rows: int, n: int, k: int, dtype) -> int:
    """Strips of 16 weight rows per workgroup of the tile kernel for a plain bf16 product that takes it without trials, 0 where trials
    decide.  A trial times candidates on whatever the memory-side cache holds and beside the launches' own time: for qkv of 64 rows
    at Qwen3-8B sizes two processes of five settled on the library's kernel (four steps 6,480 us instead of 6,320).  Weights read
    from memory, replayed, us of the tile kernel with 2 and with 4 strips and of the library's best of 16:
    N, K             20 rows            32 rows            48 rows            64 rows
    4,096, 1,024    4.8  6.0  6.3     5.0  6.3  5.5     5.6  6.8  6.4     6.2  7.5  6.8
    4,096, 2,048    7.1  9.7  8.8     7.1  9.7  8.9     8.2 10.8 12.0     9.3 11.7  9.9
    4,096, 2,560    7.9 11.1 10.1     8.6 11.7  9.5    10.1 13.1 10.5    11.1 14.4 10.6
    4,096, 4,096   11.0 15.9 13.3    12.3 16.6 11.9    14.2 18.6 14.0    15.9 20.4 14.1
    5,120, 1,024    4.9  6.4  6.5     5.2  6.5  5.9     5.8  7.0  6.8     6.4  7.7  6.9
    5,120, 5,120   13.8 19.9 17.5    15.4 21.5 18.0    17.8 23.8 20.8    19.8 25.9 21.7
    6,144, 2,560    8.4 11.7 11.4     9.3 12.4 11.7    10.7 13.9 13.4    11.9 15.2 13.7
    6,144, 4,096   12.2 16.6 15.0    13.4 17.5 15.4    15.4 19.7 17.7    17.0 21.6 18.1
    8,192, 2,048    7.9 11.8 13.3     8.3 12.3 10.5     9.2 13.0 13.7    10.3 13.8 12.3
    8,192, 5,120   17.2 25.6 19.8    17.2 23.2 20.2    19.7 25.7 22.9    21.4 28.2 24.9
    10,240, 2,560  14.7 14.5 16.8    15.5 13.6 16.1    18.4 15.2 18.0    20.7 16.7 18.2
    12,288, 4,096  24.8 21.9 26.1    24.9 21.2 25.3    28.5 22.9 26.2    31.5 24.8 26.7
    16,384, 1,024   8.8  9.0 14.0     9.1  8.9  9.9    10.1  9.6 13.9    10.9 10.3 11.0
    16,384, 5,120  31.2 31.3 35.1    34.1 31.4 35.1    37.3 31.7 35.9    41.2 33.8 37.5
    24,576, 2,048  19.7 25.8 25.3    21.0 26.5 24.9    22.8 26.5 25.4    25.8 28.2 25.2
    2,560, 9,728 (32, 48, 64 rows)   24.2 35.4 20.5    28.2 40.0 20.8    31.8 44.1 25.4
    so up to 64 rows it runs where K is short enough for a workgroup to walk whole and one round of workgroups holds the outputs, with tiles
    of 2 strips up to 32 outputs a compute unit and of 4 up to 64; below 20 outputs a compute unit only while K is short."""
    units = compute_units()
    if dtype != BF16 or not SKINNY_MAX_ROWS < rows <= PLAIN_TILE_MAX_ROWS or k > 5120 or not 16 * units <= n <= 64 * units:
        return 0
    if n < 20 * units and k > 2048:
        return 0  # o of Qwen3-8B sizes: the library's from 32 rows on
    return 2 if n <= 32 * units else 4


def _gated_tile_strips(rows: int, outputs: int) -> int:
    """Strips of 16 weight rows (gate and up together) per workgroup of the gated tile kernel: a
    workgroup loads 16 rows of weights per strip and `rows` rows of activations, and the workgroups
    run in rounds of one per compute unit; the width with the least to load on the longest path."""
    def cost(strips):
        tiles = -(-outputs // (8 * strips))
        return -(-tiles // compute_units()) * (16 * strips + rows)

    return min((8, 6, 4, 2), key=cost)


def gemm_split_plan(rows: int, n: int, k: int, dtype):
    """(strips, splits) of `gemm_split` for a product of these sizes, or None where it has no kernel:
    tiles of 64 weight rows, and K cut into as many ranges (of whole chunks, as equal as they come) as
    fill the compute units with those tiles."""
    if not _tile_rows(rows, k, dtype, TILE_SPLIT_MAX_ROWS) or n % 4:
        return None
    strips = 4
    tiles = -(-n // (16 * strips))
    chunks = k // TILE_CHUNK
    want = max(1, min(chunks, compute_units() // tiles))
    per = -(-chunks // want)  # chunks of a range; the last range may have fewer (38 chunks in 6 ranges: 7, 7, 7, 7, 7, 3)
    return strips, -(-chunks // per)


def gemm_split(a, w, plan=None):
    """The fp32 partial sums [splits, M, N] of a[M, K] @ w[N, K]^T with K cut into `splits` ranges;
    whoever takes them adds them up (`rmsnorm(..., split_sums=)`).  bf16, 17 to 128 rows."""
    _check(a, "a", BF16, (None, None))
    M, K = a.shape
    rows = _rows(w)
    _check(rows, "w", BF16, (None, K))
    N = rows.shape[0]
    plan = plan or gemm_split_plan(M, N, K, a.dtype)
    if plan is None:
        raise KernelError(f"gemm_split: {M} rows, {K} -> {N} have no kernel")
    strips, splits = plan
    sums = torch.empty((splits, M, N), dtype=F32, device=a.device)
    call("as_gemm_bf16_tile", _ptr(a), _ptr(rows), _wave_ptr(w), 0, _ptr(sums), _DT[F32], M, N, K, 0, splits, strips, _stream())
    return sums


# ---- more than 128 rows: tiles of up to 256 x 256 outputs, both operands through LDS (`csrc/gemm_wide.hip`) ---------------
WIDE_MIN_ROWS, WIDE_MAX_ROWS = TILE_MAX_ROWS + 1, 65536
WIDE_UNIT = 64  # K comes in units of this many columns
WIDE_PLAIN, WIDE_GATED, WIDE_PARTIAL = 0, 1, 2
# (rows of a, rows of w, workgroups a compute unit, us a unit of K with all places taken, with few, us a round beside the units),
# fitted to 2,900 times: 24 products of Qwen3's six sizes, 136 to 2,409 rows, every form and 1 to 12 ranges of K (off by 5 per cent on
# average, by 25 at most; the form it chooses is within 1 per cent of the best on average)
WIDE_FORMS = ((256, 256, 1, 1.33, 0.96, 6.6), (256, 192, 1, 1.09, 0.765, 4.5), (256, 128, 1, 0.83, 0.62, 2.4),
              (192, 256, 1, 1.215, 0.825, 7.6), (128, 128, 1, 0.53, 0.375, 1.0), (128, 128, 2, 1.0, 0.52, 0.5))  # fmt: skip
WIDE_LAUNCH_US, WIDE_US_A_MB, WIDE_SPLITS = 3.0, 0.2, (2, 3, 4, 6, 8, 12)
WIDE_TWO_AT_LEAST = 0.93  # of a full round's time, once a compute unit holds two workgroups (`wide_gated_form`)
WIDE_NO_PARTIAL = 3  # the form whose partial sums are not worth making (`_wide_plan`)


def _wide_cost(form: int, tiles: int, units: int) -> float:
    """Microseconds of `tiles` tiles of `units` units of K each: whole rounds of workgroups, and what is left in a round that shares
    the memory and the power among fewer."""
    *_, each, full, few, round_us = WIDE_FORMS[form]
    rounds, rest = divmod(tiles, each * compute_units())
    share = rest / (each * compute_units())
    return WIDE_LAUNCH_US + rounds * (units * full + round_us) + ((units * (few + (full - few) * share) + round_us) if rest else 0.0)


@functools.lru_cache(maxsize=4096)
def _wide_plan(rows: int, n: int, k: int, kind: int) -> tuple:
    """(us, form, splits) of the cheapest tile for a product of these sizes (kind gated: n outputs of 2 n rows of w; partial: with K cut into
    ranges whose sums are written, and read by whoever adds them up; in one round of workgroups).  Partial sums are not made in tiles of
    192 x 256: that way out takes 508 registers where the form's others take 396, and inside prompts it lost to 256 x 256 with as many
    ranges at 58 of 59 sizes measured, by up to 77 us (5,120 outputs of K = 25,600, 1,152 rows in two ranges: 48 us slower than the
    library's whole product, which they were expected to beat)."""
    best = None
    for form, (tm, tn, each, *_) in enumerate(WIDE_FORMS):
        if kind == WIDE_PARTIAL and form == WIDE_NO_PARTIAL:
            continue
        tiles = -(-rows // tm) * -(-n // (tn // 2 if kind == WIDE_GATED else tn))
        for splits in WIDE_SPLITS if kind == WIDE_PARTIAL else (1,):
            units = -(-(k // WIDE_UNIT) // splits)
            if kind == WIDE_PARTIAL and (tiles * splits > compute_units() or (splits - 1) * units >= k // WIDE_UNIT):
                continue
            us = _wide_cost(form, tiles * splits, units)
            if kind == WIDE_PARTIAL:
                us += 2 * WIDE_US_A_MB * splits * rows * n * 4e-6
            if best is None or us < best[0]:
                best = us, form, splits
    return best


def _library_us(rows: int, n: int, k: int) -> float:
    """What the library's best kernel of 16 took for the same products (off by 7 per cent on average, by a third at most)."""
    return 5.8 + 0.66e-9 * 2 * rows * n * k + 0.11 * n * k * 2e-6 + 1.79e-3 * k


def _wide_sizes(rows: int, n: int, rows_of_w: int, k: int) -> bool:
    return (WIDE_MIN_ROWS <= rows <= WIDE_MAX_ROWS and k > 0 and k % WIDE_UNIT == 0 and n > 0 and n % 16 == 0
            and max(rows, rows_of_w) * k * 2 <= 0xF0000000)  # fmt: skip


def _wide_takes(a, w, n: int, rows_of_w: int) -> bool:
    return (a.dtype == BF16 and _wide_sizes(a.shape[0], n, rows_of_w, a.shape[1]) and a.data_ptr() % 16 == 0
            and _rows(w).data_ptr() % 16 == 0)  # fmt: skip


@functools.lru_cache(maxsize=4096)
def wide_gated_form(rows: int, outputs: int, k: int):
    """The tile of a gated product of more than 128 rows, or None where the library's product with the activation after it is expected
    to take less.  Alone, us of the library's best of 16 and the activation, and of this: 3,072 outputs of K = 1,024, 256 / 1,024 / 2,409 rows
    19.1 11.5, 24.8 17.6, 38.0 32.9; 9,728 of 2,560, 512 / 2,409 rows 61 52, 228 197; 12,288 of 4,096, 333 / 512 / 2,048 rows 75 83, 91 86,
    297 300; 25,600 of 5,120, 1,500 rows 693 604.  Inside prompts of 27 lengths at six sizes, the library with the kernel that a trial of the length
    or of the next tuned one chose: 140 of 162 go to the tile and save 10 us a layer in the middle; 12 lose, 8 us of a layer's 560 once (384 rows of
    25,600 outputs), 0 to 5 of 270 to 780 else (12,288 outputs, 300, 700 and 1,900 rows).  2,048 rows of 12,288 are even: in a trace of both the tile
    312 us and the two kernels 278 and 30, a prompt through 8 such layers 6,189 to 6,224 us and 6,223 to 6,237.  (Trials of the tuned row
    counts that time the tile beside the products with their activation decide worse: the least of 16 candidates' runs against that of one gave 44
    of these to the library, 13 of which lose 9 to 30 us by it and none saves more than 10.)
    Where a compute unit holds two workgroups of the last round, the round takes as long as a full one, or nearly (tiles in the last round and us a
    unit of K: 255 0.81, 270 0.99, 303 1.07, 510 1.15): with the mean of few and full, 353 to 384 rows of 17,408 outputs and K = 5,120 went to a
    tile that took 20 us a layer more than the two kernels (a prompt of 384 tokens through 4 such layers 1,810 us, 1,730 without)."""
    us, form, _ = _wide_plan(rows, outputs, k, WIDE_GATED)
    tm, tn, each, full, few, _ = WIDE_FORMS[form]
    places = each * compute_units()
    rest = -(-rows // tm) * -(-outputs // (tn // 2)) % places
    if rest > compute_units():
        us += k // WIDE_UNIT * max(WIDE_TWO_AT_LEAST * full - (few + (full - few) * rest / places), 0.0)
    return form if us < _library_us(rows, 2 * outputs, k) + 4.0 + 6e-6 * WIDE_US_A_MB * rows * outputs else None


@functools.lru_cache(maxsize=4096)
def wide_split_plan(rows: int, n: int, k: int):
    """(form, splits) of a product of more than 128 rows cut along K into partial sums, or None where that, the sums' reading counted, is
    not expected to take less than the library's whole product.  Inside prompts of 47 lengths at six sizes, down is cut in 194 of 282 and saves
    25 us on average, nowhere less than nothing; o is cut in 100 and saves 6, and loses 5 us once (in a spread of 25) and 2 once (of a layer's
    242).  (Up to 3 per cent more than the library's was expected to take also pays for down, for o not.)  Alone, us of the two:
    4,096 outputs of K = 12,288, 256 / 512 / 1,024 rows 52 39, 78 56, 106 95; 2,560 of 9,728, 512 / 2,048 rows 52 38, 102 95; 5,120 of
    17,408, 256 rows 129 58; 1,024 of 3,072, 256 rows 12.5 10.2.  Short products of many rows stay whole (4,096 of 4,096, 700 rows 34 37)."""
    best = _wide_plan(rows, n, k, WIDE_PARTIAL)
    if best is None or best[0] >= _library_us(rows, n, k) + 2e-6 * WIDE_US_A_MB * rows * n:
        return None
    return best[1:]


F32_NARROW = 256  # up to here a 32-bit sum is one chain, which nothing cuts
F32_GROUPS = 4  # what a 32-bit sum's order comes in above that, whatever kernel runs


def gemm_f32_split_preferred(rows: int, n: int, k: int) -> bool:
    """Whether a 32-bit product of more than 16 rows, whose sums are wanted in parts, is cut into the four groups of its
    order: while its tiles of 64 x 64 outputs are no more than the compute units (512 rows, K = 2,048: N = 2,048 30 us against
    42 whole; N = 4,096 60 against 61, which the longer reading of whoever adds the parts up outweighs)."""
    return (rows > SKINNY_MAX_ROWS and k > F32_NARROW and k % 4 == 0 and n % 4 == 0
            and -(-rows // 64) * -(-n // 64) <= compute_units())  # fmt: skip


def gemm_f32_split(a, w):
    """The partial sums [4, M, N] of the 32-bit a[M, K] @ w[N, K]^T: added up in order they are `gemm`'s result (bit for bit while no
    operand exceeds bfloat16's largest number, 3.39e38; such outputs agree within rounding)."""
    _check(a, "a", F32, (None, None))
    M, K = a.shape
    rows = _rows(w)
    _check(rows, "w", F32, (None, K))
    N = rows.shape[0]
    sums = torch.empty((F32_GROUPS, M, N), dtype=F32, device=a.device)
    call("as_gemm_f32_split", _ptr(a), _ptr(rows), _ptr(sums), M, N, K, 0, _stream())
    return sums


def gemm_split_sums(a, w, choices=None):
    """a @ w^T as partial sums for whoever adds them up, or None where the product is better made whole (or has no such kernel, or
    `choices` want its kernels tried first)."""
    M, K = a.shape
    N = _rows(w).shape[0]
    if a.dtype == F32:
        return gemm_f32_split(a, w) if gemm_f32_split_preferred(M, N, K) else None
    if _wide_takes(a, w, N, N):
        plan = wide_split_plan(M, N, K)
        if plan is None or (choices or SHARED).wants_trial(M, N, K):
            return None
        form, splits = plan
        rows = _rows(w)
        _check(a, "a", BF16, (M, K))
        _check(rows, "w", BF16, (N, K))
        sums = torch.empty((splits, M, N), dtype=F32, device=a.device)
        call("as_gemm_bf16_wide", _ptr(a), _ptr(rows), _ptr(sums), M, N, K, WIDE_PARTIAL, splits, form, _stream())
        return sums
    plan = gemm_split_plan(M, N, K, a.dtype)
    return None if plan is None else gemm_split(a, w, plan)


GATED_MAX_K = 6144  # the widest input the fused product-and-activation kernel keeps in registers


def _gated_two_tiles(rows: int, k: int, w) -> bool:
    """17 to 32 rows through the persistent gated kernel with two row tiles also where the plain products of
    such widths are the library's: it saves the activation kernel and the write and read of gate and up.
    Only for weights without a copy in wave order: with one, the gated tile product is faster at these
    widths (Qwen3-8B sizes: batch 32 5,859 -> 5,980 tokens/s, batch 24 4,659 -> 4,755)."""
    return (not _wave_ptr(w) or not _tile_rows(rows, k, BF16)) and SKINNY_MAX_ROWS < rows <= SKINNY_TWO_MAX_ROWS \
        and k <= SKINNY_TWO_MAX_K and k % 8 == 0  # fmt: skip


def gemm_silu_mul(a, w, out, choices=None) -> None:
    """out[M, I] = silu(a @ w[:I]^T) * (a @ w[I:]^T) for w[2 I, K]: the gate and up products and
    the activation.  bf16 of up to 128 rows, and of more where the large tile is expected to be the faster way
    (`wide_gated_form`): one kernel, the products rounded to bf16 before the activation exactly as the two-kernel path does; fp32 of
    more than 256 columns: one kernel, the same bits as two (333 rows, 1,024 -> 6,144: 51 us, 51 and 5 for two); otherwise the
    product, then the activation."""
    _check(a, "a", (F32, BF16), (None, None))
    M, K = a.shape
    _check(out, "out", a.dtype, (M, None))
    inter = out.shape[1]
    rows = _rows(w)
    _check(rows, "w", a.dtype, (2 * inter, K))
    if M == 0:
        return
    if a.dtype == F32 and K > F32_NARROW:
        call("as_gemm_f32_gated", _ptr(a), _ptr(rows), _ptr(out), M, inter, K, 0, _stream())
        return
    if a.dtype == BF16 and (_few_rows(M, K, inter, GATED_MAX_K, w=w) or _gated_two_tiles(M, K, w)):
        call("as_gemm_bf16_gated", _ptr(a), _ptr(rows), _wave_ptr(w), _ptr(out), M, inter, K, _stream())
        return
    if _tile_rows(M, K, a.dtype):
        call("as_gemm_bf16_tile", _ptr(a), _ptr(rows), _wave_ptr(w), _ptr(out), 0, _DT[BF16], M, inter, K, 1, 0,
             _gated_tile_strips(M, inter), _stream())  # fmt: skip
        return
    if _wide_takes(a, w, inter, 2 * inter) and out.data_ptr() % 16 == 0 and not (choices or SHARED).wants_trial(M, 2 * inter, K):
        form = wide_gated_form(M, inter, K)
        if form is not None:
            call("as_gemm_bf16_wide", _ptr(a), _ptr(rows), _ptr(out), M, inter, K, WIDE_GATED, 1, form, _stream())
            return
    gate_up = torch.empty((M, 2 * inter), dtype=a.dtype, device=a.device)
    gemm(a, w, gate_up, choices)
    silu_mul(gate_up, out)


def gemm_link_supported(rows: int, n_out: int, k: int, dtype, w=None) -> bool:
    """Whether `gemm_link` and, for its result, `gemm_scaled` exist: bf16, few rows, widths the
    kernels take (n_out is the width of the stream, which is the next product's input).  w: the
    producer's weights, if known (see `_few_rows`)."""
    if dtype != BF16 or rows <= 0 or k % 8 or n_out % 8 or n_out > GATED_MAX_K:
        return False
    if w is not None and _tile_preferred(rows, k, n_out, w):
        return False
    if rows <= SKINNY_MAX_ROWS:
        return True
    # two row tiles: the producer reads its activations once per strip of 16 outputs (whole rows
    # for every workgroup of the persistent kernel, and for every strip beyond its K), the consumer
    # keeps rows of n_out in registers in each of its workgroups
    producer_strips = -(-n_out // 16) if k > SKINNY_TWO_MAX_K else min(-(-n_out // 16), _workgroups())
    return (rows <= SKINNY_TWO_MAX_ROWS and producer_strips * rows * k * 2 <= SKINNY_TWO_MAX_ACT_BYTES
            and _few_rows(rows, n_out, 16 * _workgroups()))  # fmt: skip


def gemm_f32_link_supported(rows: int, n_out: int, k: int, x=None) -> bool:
    """Whether `gemm_link` and, for its result, `gemm_scaled` exist in 32 bits: one row tile, both products' sums in the
    order that is cut (their kernels; n_out is the width of the stream, which is the next product's input).  x: the stream, if known.
    Four decode steps of 4 requests at Qwen3-0.6B sizes: 7,824 us without, 7,258 with (the norm's kernel takes 4.4 us)."""
    return (0 < rows <= SKINNY_MAX_ROWS and k > F32_NARROW and n_out > F32_NARROW and n_out % 4 == 0
            and (x is None or x.data_ptr() % 16 == 0))  # fmt: skip


def link_strips(n: int, dtype) -> int:
    """Sums of squares that a row of n columns carries from a `gemm_link` to a `gemm_scaled`."""
    return -(-n // (4 if dtype == F32 else 16))


def gemm_link(a, w, x, gain, scaled, ssq) -> None:
    """The last product of a part of a pre-norm layer with the residual sum and the first half of
    the next RMSNorm: x[M, N] (fp32) += bf16(a @ w^T); scaled[M, N] = bf16(x * gain), the next
    product's input without its 1/rms factor; ssq[M, ceil(N / 16)] = sums of x^2 per 16 columns.
    a, w, scaled bf16, or all fp32 and nothing rounded (ssq then [M, N / 4], per 4 columns); gain fp32 [N]."""
    _check(a, "a", (F32, BF16), (None, None))
    M, K = a.shape
    rows = _rows(w)
    _check(rows, "w", a.dtype, (None, K))
    N = rows.shape[0]
    if not (gemm_f32_link_supported(M, N, K, x) if a.dtype == F32 else gemm_link_supported(M, N, K, a.dtype)):
        raise KernelError(f"gemm_link: {M} rows, {K} -> {N} have no fused kernel")
    _check(x, "x", F32, (M, N))
    _check(gain, "gain", F32, (N,))
    _check(scaled, "scaled", a.dtype, (M, N))
    _check(ssq, "ssq", F32, (M, link_strips(N, a.dtype)))
    if a.dtype == F32:
        call("as_gemm_f32_link", _ptr(a), _ptr(rows), _ptr(x), _ptr(gain), _ptr(scaled), _ptr(ssq), M, N, K, _stream())
        return
    call("as_gemm_bf16_link", _ptr(a), _ptr(rows), _wave_ptr(w), _ptr(x), _ptr(gain), _ptr(scaled), _ptr(ssq), M, N, K,
         _stream())  # fmt: skip


def gemm_scaled(scaled, ssq, eps, w, out, gated=False) -> None:
    """The first product of the part that follows a `gemm_link`: out = (scaled @ w^T) / rms with
    rms^2 = sum(ssq) / K + eps per row (gated: silu of the first half of w's rows times the
    second half, both scaled and rounded to bf16 first).  scaled [M, K], w, out bf16, or all fp32."""
    _check(scaled, "scaled", (F32, BF16), (None, None))
    M, K = scaled.shape
    _check(ssq, "ssq", F32, (M, link_strips(K, scaled.dtype)))
    _check(out, "out", scaled.dtype, (M, None))
    N = out.shape[1]
    rows = _rows(w)
    _check(rows, "w", scaled.dtype, (2 * N if gated else N, K))
    if scaled.dtype == F32:
        if not gemm_f32_link_supported(M, K, K):
            raise KernelError(f"gemm_scaled: {M} rows of width {K} have no fused kernel")
        call("as_gemm_f32_scaled", _ptr(scaled), _ptr(ssq), ssq.shape[1], float(eps), _ptr(rows), _ptr(out), M, N, K,
             int(bool(gated)), _stream())  # fmt: skip
        return
    if not gemm_link_supported(M, K, 8, BF16):
        raise KernelError(f"gemm_scaled: {M} rows of width {K} have no fused kernel")
    call("as_gemm_bf16_scaled", _ptr(scaled), _ptr(ssq), ssq.shape[1], float(eps), _ptr(rows), _wave_ptr(w), _ptr(out), M, N, K,
         int(bool(gated)), _stream())  # fmt: skip


SAMPLE_MAX_TOP_K = 1024


def argmax(logits, out) -> None:
    """out[b] = index of the largest logit of row b (the lowest index among equals)."""
    _check(logits, "logits", F32, (None, None))
    _check(out, "out", I32, (logits.shape[0],))
    call("as_argmax", _ptr(logits), _ptr(out), logits.shape[0], logits.shape[1], _stream())


def apply_penalty(logits, rows, cols, amounts) -> None:
    """logits[rows[i], cols[i]] -= amounts[i] for distinct (row, col) pairs."""
    _check(logits, "logits", F32, (None, None))
    n = rows.shape[0]
    _check(rows, "rows", I32, (n,))
    _check(cols, "cols", I32, (n,))
    _check(amounts, "amounts", F32, (n,))
    call("as_apply_penalty", _ptr(logits), _ptr(rows), _ptr(cols), _ptr(amounts), n, logits.shape[1], _stream())


SAMPLE_SPLIT_MAX_TOP_K = 64  # up to here a row's candidates are found by 32 workgroups instead of one


def sample(logits, temperature, top_k, top_p, seeds, counters, out, max_top_k=None) -> None:
    """One token per row: top-k (0: all), temperature (0: greedy), top-p, seeded draw.

    temperature, top_p fp32 [B]; top_k, counters int32 [B]; seeds int64 [B]; out int32 [B].
    A top_k of 0 (or >= vocabulary) keeps all tokens; up to SAMPLE_MAX_TOP_K the candidates are
    ranked (the lower index first among equals); beyond, every token at least as large as the k-th
    largest stays (equal ones together).  max_top_k: the caller's promise that every row keeps between 1
    and this many candidates (a greedy row keeps 1); up to SAMPLE_SPLIT_MAX_TOP_K the rows are
    then searched by many workgroups each, with the same result."""
    _check(logits, "logits", F32, (None, None))
    B = logits.shape[0]
    _check(temperature, "temperature", F32, (B,))
    _check(top_k, "top_k", I32, (B,))
    _check(top_p, "top_p", F32, (B,))
    _check(seeds, "seeds", torch.int64, (B,))
    _check(counters, "counters", I32, (B,))
    _check(out, "out", I32, (B,))
    if max_top_k is not None and 1 <= max_top_k <= SAMPLE_SPLIT_MAX_TOP_K:
        cand = torch.empty((B, 32, SAMPLE_SPLIT_MAX_TOP_K), dtype=torch.int64, device=logits.device)
        counts = torch.empty((B, 32), dtype=I32, device=logits.device)
        call("as_sample_split", _ptr(logits), B, logits.shape[1], _ptr(temperature), _ptr(top_k), _ptr(top_p),
             _ptr(seeds), _ptr(counters), _ptr(cand), _ptr(counts), _ptr(out), _stream())  # fmt: skip
        return
    call("as_sample", _ptr(logits), B, logits.shape[1], _ptr(temperature), _ptr(top_k), _ptr(top_p), _ptr(seeds),
         _ptr(counters), _ptr(out), _stream())  # fmt: skip


def topk(logits, k, values, indices) -> None:
    """Sorted k largest of each row: values fp32 [B, k], indices int32 [B, k]."""
    _check(logits, "logits", F32, (None, None))
    B, V = logits.shape
    if not 0 < k <= min(V, SAMPLE_MAX_TOP_K):
        raise KernelError(f"top-k of {k} is outside 1..{min(V, SAMPLE_MAX_TOP_K)}")
    _check(values, "values", F32, (B, k))
    _check(indices, "indices", I32, (B, k))
    call("as_topk", _ptr(logits), B, V, k, _ptr(values), _ptr(indices), _stream())


# ---- sublayers whose output is normed before it enters the stream ----------------------------------------------------


def post_norm_add(x, y, post, eps_post, gain=None, eps: float = 0.0, out=None, rows=None, update_x=True, other=None, gains=None,
                  biases=(None, None), eps_in: float = 0.0, centre_post: bool = False, centre: bool = False) -> None:  # fmt: skip
    """v = x[s] + norm(d[s]) * post with s = rows[r] or r (eps_post inside the root), x fp32 [T, n] receiving v when
    `update_x`; out[r] = norm(v) * gain (gain None: no norm is taken, and out, if there is one, receives v itself).
    centre_post, centre: that norm takes the row's mean off first (a layer norm without a bias).  d = y (+ biases[0]); with `other`, d =
    norm(y + biases[0]) * gains[0] + norm(other + biases[1]) * gains[1] (eps_in).  y, other [T, n] and out in the compute
    dtype; post, gain, gains and biases fp32 [n]."""
    _check(x, "x", F32, (None, None))
    T, n = x.shape
    _check(y, "y", (F32, BF16), (T, n))
    n_out = T
    if rows is not None:
        _check(rows, "rows", I32, (None,))
        n_out = rows.shape[0]
        if update_x:
            raise KernelError("post_norm_add: the stream is updated whole, not by rows")
    if gain is not None and out is None:
        raise KernelError("post_norm_add: a norm's gain comes with its output")
    for name, t in (("post", post), ("gain", gain), ("bias", biases[0]), ("other bias", biases[1])):
        if t is not None or name == "post":
            _check(t, name, F32, (n,))
    if out is not None:
        _check(out, "out", y.dtype, (n_out, n))
    g1 = g2 = None
    if other is not None:
        _check(other, "other", y.dtype, (T, n))
        g1, g2 = gains
        _check(g1, "gain of y", F32, (n,))
        _check(g2, "gain of other", F32, (n,))
    elif biases[1] is not None:
        raise KernelError("post_norm_add: a second bias belongs to a second output")
    call("as_post_norm_add", _ptr(x), _ptr(y), _ptr(other), _DT[y.dtype], _ptr(biases[0]), _ptr(biases[1]), _ptr(g1), _ptr(g2),
         float(eps_in), _ptr(post), float(eps_post), _ptr(gain), float(eps), int(bool(centre_post)),
         int(bool(centre)), _ptr(rows), _ptr(out), n_out, n, int(bool(update_x)), _stream())  # fmt: skip


def layer_norm(x, gain, eps, out, delta=None, rows=None, update_x=True) -> None:
    """v = x[s] (+ delta[s]) with s = rows[r] or r, x fp32 [T, n] receiving v when something was added and `update_x`;
    out[r] = (v - mean) / sqrt(mean((v - mean)^2) + eps) * gain, gain fp32 [n]; delta [T, n] of out's dtype or None."""
    _check(x, "x", F32, (None, None))
    T, n = x.shape
    _check(gain, "gain", F32, (n,))
    n_out = T
    if rows is not None:
        _check(rows, "rows", I32, (None,))
        n_out = rows.shape[0]
        if update_x and delta is not None:
            raise KernelError("layer_norm: the stream is updated whole, not by rows")
    _check(out, "out", (F32, BF16), (n_out, n))
    if delta is not None:
        _check(delta, "delta", out.dtype, (T, n))
    call("as_layer_norm", _ptr(x), _ptr(delta), _ptr(gain), float(eps), _ptr(rows), _ptr(out), _DT[out.dtype], n_out, n,
         int(bool(update_x)), _stream())  # fmt: skip


def token_gate(z, table, ids, out) -> None:
    """out[t] = gelu(z[t]) * table[ids[t]] (the tanh form of gelu): z, out [T, dim], table [vocab, dim], ids int32 [T]."""
    _check(z, "z", (F32, BF16), (None, None))
    T, dim = z.shape
    _check(table, "table", z.dtype, (None, dim))
    _check(ids, "ids", I32, (T,))
    _check(out, "out", z.dtype, (T, dim))
    call("as_token_gate", _ptr(z), _ptr(table), _ptr(ids), _DT[z.dtype], _ptr(out), dim, T, _stream())


TOKEN_PRODUCT_MAX_ROWS = 16


def gemm_token_gate(x, w, table, ids, out, choices=None) -> None:
    """out[t] = gelu(x[t] @ w^T) * table[ids[t]]: x [T, K], w [dim, K] (or its `Streamed`), table [vocab, dim], out [T, dim].
    Few rows in one kernel (every product's sum in fp32 until the gate), more as a product and `token_gate`."""
    rows = _rows(w)
    _check(x, "x", (F32, BF16), (None, None))
    T, K = x.shape
    dim = rows.shape[0]
    if x.dtype == BF16 and T <= TOKEN_PRODUCT_MAX_ROWS and K % 8 == 0:
        _check(rows, "w", BF16, (dim, K))
        _check(table, "table", BF16, (None, dim))
        _check(ids, "ids", I32, (T,))
        _check(out, "out", BF16, (T, dim))
        call("as_token_product", _ptr(x), _ptr(rows), _ptr(table), _ptr(ids), _ptr(out), K, dim, T, _stream())
        return
    z = torch.empty((T, dim), dtype=x.dtype, device=x.device)
    gemm(x, w, z, choices)
    token_gate(z, table, ids, out)


def poly_norm(z, coef, eps, out) -> None:
    """out = a N(z) + b N(z^2) + c N(z^3) + e per row, N the division by the row's root mean square (eps inside the root);
    coef fp32 [4] = a, b, c, e."""
    _check(z, "z", (F32, BF16), (None, None))
    _check(coef, "coef", F32, (4,))
    _check(out, "out", z.dtype, tuple(z.shape))
    call("as_poly_norm", _ptr(z), _DT[z.dtype], _ptr(coef), float(eps), _ptr(out), z.shape[0], z.shape[1], _stream())


# ---- layers whose parts read one stream side by side -------------------------------------------------


def rmsnorm_multi(x, weight1, weight2, eps, out1, out2=None, delta1=None, delta2=None, rows=None, update_x=True) -> None:
    """v = x[s] + (delta1[s] + delta2[s]) (either may be absent), s = rows[r] or r; out1[r] = norm(v) * weight1 and,
    if given, out2[r] = norm(v) * weight2, the root mean square taken once; x fp32 [T, n] receives v when
    `update_x` and something was added."""
    _check(x, "x", F32, (None, None))
    T, n = x.shape
    n_out = T
    if rows is not None:
        _check(rows, "rows", I32, (None,))
        n_out = rows.shape[0]
    _check(out1, "out1", (F32, BF16), (n_out, n))
    _check(weight1, "weight1", (F32, BF16), (n,))
    if out1.dtype == F32 and weight1.dtype != F32:
        raise KernelError("fp32 norm needs an fp32 weight")
    if (out2 is None) != (weight2 is None):
        raise KernelError("a second output and a second weight come together")
    if out2 is not None:
        _check(out2, "out2", out1.dtype, (n_out, n))
        _check(weight2, "weight2", weight1.dtype, (n,))
    for name, d in (("delta1", delta1), ("delta2", delta2)):
        if d is not None:
            _check(d, name, out1.dtype, (T, n))
    call("as_rmsnorm_multi", _ptr(x), _ptr(delta1), _ptr(delta2), _ptr(rows), _ptr(weight1), _ptr(weight2),
         _DT[weight1.dtype], float(eps), _ptr(out1), _ptr(out2), _DT[out1.dtype], n_out, n, int(bool(update_x)), _stream())  # fmt: skip


def head_norm_store(proj, q_off, k_off, v_off, num_heads, num_kv_heads, dim, vdim, q_weight, k_weight, eps, slots,
                    q_out, k_pages, v_pages, store_kv=True, cos_sin=None) -> None:  # fmt: skip
    """Heads cut out of a wider projection's output proj [T, ld] (queries at column q_off, keys at k_off, both
    `dim` wide; values at v_off, `vdim` wide): per-head RMS norm of queries and keys (weights [dim], or none), their
    rotation where `cos_sin` (fp32 [T, R/2, 2]) is given (the pairs (i, i + R/2) of a head's first R coordinates;
    values are never turned, so v_off = k_off stores the unturned keys as values), and the cache store.  Every head is laid out Dp = q_out.shape[2] >= max(dim, vdim) wide, zero where
    it has no coordinate: q_out [T, H, Dp], k_pages [pages, KV, bs, Dp], v_pages [pages, KV, Dp, bs]."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    H, KV = num_heads, num_kv_heads
    _check(q_out, "q_out", proj.dtype, (T, H, None))
    Dp = q_out.shape[2]
    if Dp < max(dim, vdim) or min(q_off, k_off, v_off) < 0 or q_off + H * dim > ld or k_off + KV * dim > ld \
            or v_off + KV * vdim > ld:  # fmt: skip
        raise KernelError("head_norm_store: heads lie outside the projection's columns or the padded head width")
    w_dtype = proj.dtype
    if q_weight is not None:
        _check(q_weight, "q_weight", (F32, BF16), (dim,))
        _check(k_weight, "k_weight", q_weight.dtype, (dim,))
        w_dtype = q_weight.dtype
        if proj.dtype == F32 and w_dtype != F32:
            raise KernelError("fp32 q/k norm needs fp32 weights")
    elif k_weight is not None:
        raise KernelError("q and k norm weights come together")
    bs = 1
    if store_kv:
        _check(slots, "slots", I32, (T,))
        _check(k_pages, "k_pages", proj.dtype, (None, KV, None, Dp))
        bs = k_pages.shape[2]
        _check(v_pages, "v_pages", proj.dtype, (k_pages.shape[0], KV, Dp, bs))
    R = 0
    if cos_sin is not None:
        _check(cos_sin, "cos_sin", F32, (T, None, 2))
        R = 2 * cos_sin.shape[1]
        if R > dim or R < 2:
            raise KernelError(f"head_norm_store: {R} turned coordinates in a head of {dim}")
    call("as_head_norm_store", _ptr(proj), _DT[proj.dtype], ld, q_off, k_off, v_off, H, KV, dim, vdim, Dp,
         _ptr(q_weight), _ptr(k_weight), _DT[w_dtype], float(eps), _ptr(slots) if store_kv else 0, _ptr(q_out),
         _ptr(k_pages) if store_kv else 0, _ptr(v_pages) if store_kv else 0, bs, int(bool(store_kv)), T,
         _ptr(cos_sin), R, _stream())  # fmt: skip


def whole_norm_store(proj, q_off, k_off, v_off, num_heads, num_kv_heads, dim, vdim, slots, q_out, k_pages, v_pages,
                     store_kv=True, biases=None, gains=None, eps: float = 0.0, cos_sin=None, v_keep=None,
                     v_mode: str = "none", lam: float = 0.0, maps: int = 1) -> None:  # fmt: skip
    """`head_norm_store` for heads that are normed over their whole projection.  biases: (q [H dim], k [KV dim], v [KV
    vdim]) fp32, added to the projection's output first, or None.  gains: (q [H dim], k [KV dim]) fp32: queries and keys
    are divided by the root mean square over ALL their heads (eps inside the root) and multiplied by the gains (k None: the
    queries alone, without keys to store); None: no norm.  cos_sin: the rotation (after the norm), as in `head_norm_store`.  v_mode "keep": the values (bias added) are
    also written to v_keep fp32 [T, KV vdim]; "mix": (1 - lam) v + lam v_keep[t] is stored instead of v.
    maps > 1: every head has that many queries and keys over the same values.  num_heads counts the queries (heads x
    maps, `dim` / maps wide each in proj), dim is all of a head's keys side by side, and a query is laid out at its map's
    place among them, zeros elsewhere; no norm and no rotation.  store_kv off: proj need not hold keys and values."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    H, KV = num_heads, num_kv_heads
    _check(q_out, "q_out", proj.dtype, (T, H, None))
    Dp = q_out.shape[2]
    if maps < 1 or dim % maps or H % maps or (maps > 1 and (gains is not None or cos_sin is not None)):
        raise KernelError(f"whole_norm_store: {maps} maps of {dim} coordinates in all, {H} queries, no norm and no rotation")
    if Dp < max(dim, vdim) or q_off < 0 or q_off + H * (dim // maps) > ld or \
            ((store_kv or (gains is not None and gains[1] is not None) or v_mode != "none") and
             (min(k_off, v_off) < 0 or k_off + KV * dim > ld or v_off + KV * vdim > ld)):  # fmt: skip
        raise KernelError("whole_norm_store: heads lie outside the projection's columns or the padded head width")
    qb = kb = vb = qw = kw = inverse = None
    if biases is not None:
        qb, kb, vb = biases
        for name, t, n in (("q bias", qb, H * (dim // maps)), ("k bias", kb, KV * dim), ("v bias", vb, KV * vdim)):
            if t is not None or store_kv or name == "q bias":
                _check(t, name, F32, (n,))
    if gains is not None:
        qw, kw = gains
        _check(qw, "q gain", F32, (H * dim,))
        if kw is not None or store_kv:
            _check(kw, "k gain", F32, (KV * dim,))
        if proj.dtype == BF16 and not (ld | q_off | k_off | v_off | dim | vdim | Dp) & 7:
            # the root mean squares first, then 16 bytes of a head a thread
            inverse = torch.empty((T, 2), dtype=F32, device=proj.device)
    bs = 1
    if store_kv:
        _check(slots, "slots", I32, (T,))
        _check(k_pages, "k_pages", proj.dtype, (None, KV, None, Dp))
        bs = k_pages.shape[2]
        _check(v_pages, "v_pages", proj.dtype, (k_pages.shape[0], KV, Dp, bs))
    R = 0
    if cos_sin is not None:
        _check(cos_sin, "cos_sin", F32, (T, None, 2))
        R = 2 * cos_sin.shape[1]
        if R > dim or R < 2:
            raise KernelError(f"whole_norm_store: {R} turned coordinates in a head of {dim}")
    modes = {"none": 0, "keep": 1, "mix": 2}
    if v_mode not in modes:
        raise KernelError(f"whole_norm_store: values are handled as one of {sorted(modes)}, not {v_mode!r}")
    if modes[v_mode]:
        _check(v_keep, "v_keep", F32, (T, KV * vdim))
    call("as_whole_norm_store", _ptr(proj), _DT[proj.dtype], ld, q_off, k_off, v_off, H, KV, dim, vdim, Dp, _ptr(qb),
         _ptr(kb), _ptr(vb), _ptr(qw), _ptr(kw), float(eps), _ptr(inverse), _ptr(cos_sin), R, _ptr(v_keep) if modes[v_mode] else 0,
         modes[v_mode], float(lam), _ptr(slots) if store_kv else 0, _ptr(q_out), _ptr(k_pages) if store_kv else 0,
         _ptr(v_pages) if store_kv else 0, bs, int(bool(store_kv)), int(maps), T, _stream())  # fmt: skip


def map_difference(heads, vdim, lam, eps, mult, out, out_off: int = 0) -> None:
    """heads [T, 2 H, Dp] (out's dtype, or fp32): head h's two attention maps at 2 h and 2 h + 1, `vdim` coordinates wide.  With o = a1 - lam a2:
    out[t, out_off + h * vdim + j] = mult * o_j / sqrt(mean(o^2) + eps)."""
    _check(heads, "heads", (F32, BF16), (None, None, None))
    T, H2, Dp = heads.shape
    _check(out, "out", (F32, BF16) if heads.dtype == F32 else BF16, (T, None))
    if H2 % 2 or not 1 <= vdim <= Dp or out_off < 0 or out_off + H2 // 2 * vdim > out.shape[1]:
        raise KernelError(f"map_difference: {H2} maps of {Dp} coordinates, {vdim} of them values, columns {out_off}.. of {out.shape[1]}")
    call("as_map_difference", _ptr(heads), _DT[heads.dtype], H2 // 2, vdim, Dp, float(lam), float(eps), float(mult), _ptr(out),
         _DT[out.dtype], out.shape[1], out_off, T, _stream())  # fmt: skip


STREAMS_MAX = 16


def streams_step(xs, first=None, y=None, mix=None, out_c=None, mult: float = 1.0, in_c=None, gain=None, eps: float = 0.0,
                 normed=None, total=None) -> None:  # fmt: skip
    """One step between two parts of a model with several residual streams xs fp32 [T, S, n] (updated in place).
    first [T, n] fp32: the streams do not exist yet, all of them are `first`.  y [T, n] (compute dtype): the pending
    write xs[:, r] <- sum_s mix[s, r] xs[:, s] + mult out_c[r] y (mix fp32 [S, S], None: the identity; out_c fp32 [S]).
    in_c fp32 [S] with gain fp32 [n] and normed [T, n] (compute dtype): normed = rmsnorm(sum_s in_c[s] xs[:, s]) * gain.
    total fp32 [T, n]: receives sum_s xs[:, s]."""
    _check(xs, "xs", F32, (None, None, None))
    T, S, n = xs.shape
    if not 1 <= S <= STREAMS_MAX:
        raise KernelError(f"1 to {STREAMS_MAX} streams, not {S}")
    dtype = None
    if first is not None:
        _check(first, "first", F32, (T, n))
    if y is not None:
        _check(y, "y", (F32, BF16), (T, n))
        dtype = y.dtype
        _check(out_c, "out_c", F32, (S,))
        if mix is not None:
            _check(mix, "mix", F32, (S, S))
    if (in_c is None) != (normed is None):
        raise KernelError("streams_step: the read's weights and the normed rows come together")
    if normed is not None:
        _check(normed, "normed", (F32, BF16) if dtype is None else dtype, (T, n))
        dtype = normed.dtype
        _check(in_c, "in_c", F32, (S,))
        _check(gain, "gain", F32, (n,))
    if total is not None:
        _check(total, "total", F32, (T, n))
    call("as_streams_step", _ptr(xs), _ptr(first), S, n, _ptr(y), _DT[dtype if dtype is not None else F32], _ptr(mix),
         _ptr(out_c), float(mult), _ptr(in_c), _ptr(gain), float(eps), _ptr(normed), _ptr(total), T, _stream())  # fmt: skip


def gated_add_norm(x, y, gate, gate_off, bias, mult, weight, eps, out, rows=None, update_x=True, other=None,
                   join=None) -> None:  # fmt: skip
    """The fp32 stream x [T, n] takes a part's gated, scaled output and is normed, in one kernel:
    x[s] += mult * sigmoid(gate[s, gate_off:gate_off + n] + bias) * y[s]   (y None: nothing is added)
    out[r] = x[s] / sqrt(mean(x[s]^2) + eps) * weight                      (weight None: no norm; out fp32 or y's dtype)
    join[r] = [x[s] | other[s]] in the compute dtype                        (join None: none)
    with s = rows[r] (or r).  y [T, n] and gate [T, ld] are a part's output and the logits of its gate."""
    _check(x, "x", F32, (None, None))
    T, n = x.shape
    n_out = T
    if rows is not None:
        _check(rows, "rows", I32, (None,))
        n_out = rows.shape[0]
    dtype = None
    ld = 0
    if y is not None:
        _check(y, "y", (F32, BF16), (T, n))
        dtype = y.dtype
        _check(gate, "gate", dtype, (T, None))
        ld = gate.shape[1]
        if gate_off < 0 or gate_off + n > ld:
            raise KernelError("gated_add_norm: the gate lies outside its product's columns")
    if join is not None:
        _check(join, "join", (F32, BF16) if dtype is None else dtype, (n_out, 2 * n))
        _check(other, "other", F32, (T, n))
        dtype = join.dtype
    w_dtype = None
    for name, v in (("weight", weight), ("bias", bias)):
        if v is not None:
            _check(v, name, (F32, BF16) if w_dtype is None else w_dtype, (n,))
            w_dtype = v.dtype
    if weight is not None:
        _check(out, "out", (F32, BF16), (n_out, n))
        if dtype is None:
            dtype = out.dtype if out.dtype == BF16 else weight.dtype
    if dtype is None:
        return  # nothing to add, to norm or to join
    if w_dtype is None:
        w_dtype = dtype
    if dtype == F32 and w_dtype != F32:
        raise KernelError("gated_add_norm: 32-bit rows need 32-bit gains and biases")
    out_dtype = out.dtype if weight is not None else dtype
    call("as_gated_add_norm", _ptr(x), _ptr(y), _ptr(gate), _DT[dtype], ld, gate_off, _ptr(bias), float(mult),
         _ptr(rows), _ptr(weight), _DT[w_dtype], float(eps), _ptr(out) if weight is not None else 0, _DT[out_dtype],
         n_out, n, int(bool(update_x)), _ptr(other), _ptr(join), _stream())  # fmt: skip


def relu2(a, off, out) -> None:
    """out[t, i] = max(a[t, off + i], 0)^2 for the out.shape[1] columns of a [T, ld] from `off` on."""
    _check(a, "a", (F32, BF16), (None, None))
    T, ld = a.shape
    _check(out, "out", a.dtype, (T, None))
    n = out.shape[1]
    if off < 0 or off + n > ld:
        raise KernelError("relu2: columns outside the input")
    call("as_relu2", _ptr(a), _DT[a.dtype], ld, off, _ptr(out), n, T, _stream())


# ---- attention with mixed heads ----------------------------------------------------------------------

HEADMIX_KEYS = 64  # key slots of a chunk
HEADMIX_MAX_LDS = 96 << 10


def attn_headmix_tile(num_heads: int, head_dim: int, dtype) -> int:
    """The most consecutive queries of a row that one workgroup of `attn_headmix` takes (16, 8, 4, 2 or 1):
    bounded by the accumulators a thread keeps and by LDS; 0: the kernel does not take so many heads."""
    elt = 4 if dtype == F32 else 2
    for tile, most in ((16, 4), (8, 8), (4, 16), (2, 32), (1, 32)):
        if -(-num_heads * head_dim // 256) > most:
            continue
        floats = 2 * num_heads * tile * HEADMIX_KEYS + num_heads * num_heads + 3 * tile * num_heads + HEADMIX_KEYS
        if floats * 4 + 16 + tile * num_heads * head_dim * elt > HEADMIX_MAX_LDS:
            continue
        return tile
    return 0


HEADMIX_MFMA_MAX_LDS = 128 << 10
HEADMIX_MFMA_TILES = 16  # output tiles (kv head, 64 coordinates) that a wave of the matrix-core kernel keeps
HEADMIX_FILL = 2  # workgroups per compute unit up to which an item's keys are cut over several workgroups
HEADMIX_MAX_SPLITS = 64


def _headmix_mfma_lds(H: int, D: int, tq: int) -> int:
    h8 = -(-H // 8) * 8
    scores = -(-H * tq * (HEADMIX_KEYS + 1) // 4) * 4  # rows a little longer than their 64 slots, against bank conflicts
    return (scores + H * h8 + 3 * tq * H + HEADMIX_KEYS) * 4 + 16 + (H * tq * (HEADMIX_KEYS + 8) + tq * H * (D + 8)) * 2


def attn_headmix_mfma_takes(dtype, H: int, KV: int, D: int, block_size: int, tile: int) -> bool:
    """Whether the matrix-core form of `attn_headmix` takes these sizes with items of up to `tile` queries: bf16,
    heads of 32, 64, 96, 128, 192 or 256 coordinates, `tile` queries times the heads of a kv head within a tile's 16 rows,
    pages of 8, 16, 32 or 64 tokens."""
    if dtype != BF16 or H < 1 or KV < 1 or H % KV or H > 64 or tile < 1 or (H // KV) * tile > 16:
        return False
    if (H // KV) & (H // KV - 1):  # 1, 2, 4, 8 or 16 query heads to a kv head: the rows of a tile are cut by shifts
        return False
    if D not in (32, 64, 96, 128, 192, 256) or KV * -(-D // 64) > HEADMIX_MFMA_TILES:
        return False
    if block_size % 8 or block_size > HEADMIX_KEYS or HEADMIX_KEYS % block_size:
        return False
    return _headmix_mfma_lds(H, D, tile) <= HEADMIX_MFMA_MAX_LDS


def attn_headmix_rows(num_heads: int, num_kv_heads: int, head_dim: int, dtype) -> int:
    """How many consecutive queries of a row make a work item of `attn_headmix` for a model of these sizes: what the
    matrix-core kernel packs into a tile's 16 rows beside the heads of a kv head, where it takes the sizes at all
    (whatever the pages: the general kernel serves the pages it does not, taking such an item in turns); else what
    the general kernel takes at once."""
    if attn_headmix_mfma_takes(dtype, num_heads, num_kv_heads, head_dim, 16, 1):
        tile = 16
        while tile > 1 and not attn_headmix_mfma_takes(dtype, num_heads, num_kv_heads, head_dim, 16, tile):
            tile //= 2
        return tile
    return attn_headmix_tile(num_heads, head_dim, dtype)


def _headmix_splits(num_items: int, tile: int, window: int, keep_first: int, max_context: int) -> int:
    """Into how many workgroups an item's keys are cut: one where the items alone fill the GPU, else as many as fill
    it, each with at least one chunk of 64 keys."""
    if max_context <= 0:
        return 1
    keys = max_context if window <= 0 else min(max_context, window + tile - 1 + keep_first + HEADMIX_KEYS)
    chunks = -(-keys // HEADMIX_KEYS) + 1
    want = -(-HEADMIX_FILL * compute_units() // max(1, num_items))
    return max(1, min(chunks, want, HEADMIX_MAX_SPLITS))


def attn_headmix(q, k_pages, v_pages, items, tile: int, positions, tok_row, block_tables, mix, out, scale: float,
                 window: int = 0, keep_first: int = 0, max_context: int = 0, splits: int = None) -> None:  # fmt: skip
    """Softmax attention whose heads' scores are mixed before the softmax: s_h = sum_g mix[h, g] * scale * q_g . k
    (mix fp32 [H, H]; None: no mixing), a query at position i seeing the keys j <= i with i - j < window (0: all)
    or j < keep_first.  q [T, H, D]; out [T, H, Dout], Dout <= D (heads padded to D with zeros lose the padding);
    pages as the other attention kernels read them.
    tile == 1: items [N] int32 are single tokens (positions [T]; tok_row [T] or None where token t is row t);
    else items [N, 4] = (first token, count <= tile, row, first position).
    bf16 with sizes that `attn_headmix_mfma_takes` runs on the matrix cores; max_context (a bound on the positions,
    0: unknown) lets few items' keys be cut over several workgroups (`splits`: forced, for tests)."""
    _check(q, "q", (F32, BF16), (None, None, None))
    T, H, D = q.shape
    _check(out, "out", q.dtype, (T, H, None))
    Dout = out.shape[2]
    if not 1 <= Dout <= D:
        raise KernelError(f"attn_headmix: outputs of {Dout} coordinates from heads of {D}")
    _check(k_pages, "k_pages", q.dtype, (None, None, None, D))
    NB, KV, bs, _ = k_pages.shape
    _check(v_pages, "v_pages", q.dtype, (NB, KV, D, bs))
    _check(block_tables, "block_tables", I32, (None, None))
    if H % KV or bs > HEADMIX_KEYS:
        raise KernelError(f"attn_headmix: {H} heads over {KV} kv heads, pages of {bs} (at most {HEADMIX_KEYS})")
    if D % (4 if q.dtype == F32 else 8):
        raise KernelError(f"attn_headmix: heads of {D} are not read 16 bytes at a time")
    if tile not in (1, 2, 4, 8, 16):
        raise KernelError(f"attn_headmix: a tile of {tile} queries (1, 2, 4, 8 or 16)")
    mfma = attn_headmix_mfma_takes(q.dtype, H, KV, D, bs, tile)
    if not mfma and attn_headmix_tile(H, D, q.dtype) < 1:  # (an item of more queries than fit at once is taken in turns)
        raise KernelError(f"attn_headmix: {H} heads of {D} are more than a workgroup keeps at once")
    if tile == 1:
        _check(items, "items", I32, (None,))
        _check(positions, "positions", I32, (T,))
        if tok_row is not None:
            _check(tok_row, "tok_row", I32, (T,))
    else:
        _check(items, "items", I32, (None, 4))
    if mix is not None:
        _check(mix, "mix", F32, (H, H))
    if window < 0 or keep_first < 0:
        raise KernelError("attn_headmix: a window and a number of kept tokens are not negative")
    if mfma:
        N = items.shape[0]
        if splits is None:
            splits = _headmix_splits(N, tile, window, keep_first, max_context)
        part_o = part_ml = None
        if splits > 1:
            part_o = torch.empty((N, splits, tile, H, D), dtype=F32, device=q.device)
            part_ml = torch.empty((N, splits, tile, H, 2), dtype=F32, device=q.device)
        call("as_attn_headmix_mfma", _ptr(q), _ptr(k_pages), _ptr(v_pages), _ptr(items), N, tile, int(tile == 1),
             _ptr(positions), _ptr(tok_row), _ptr(block_tables), block_tables.shape[1], _ptr(mix), _ptr(out), H, KV, D,
             Dout, bs, float(scale), int(window), int(keep_first), int(splits), _ptr(part_o), _ptr(part_ml), _stream())  # fmt: skip
        return
    call("as_attn_headmix", _ptr(q), _ptr(k_pages), _ptr(v_pages), _DT[q.dtype], _ptr(items), items.shape[0], tile,
         _ptr(positions), _ptr(tok_row), _ptr(block_tables), block_tables.shape[1], _ptr(mix), _ptr(out), H, KV, D,
         Dout, bs, float(scale), int(window), int(keep_first), _stream())  # fmt: skip


def sigmoid_gate_heads(heads, vdim, gate, gate_off, scale, out, out_off, per_head: bool = False) -> None:
    """out[t, out_off + h * vdim + j] = scale * sigmoid(gate[t, gate_off + h * vdim + j]) * heads[t, h, j], j < vdim;
    gate None: scale * heads, laid side by side; per_head: one number a head, gate[t, gate_off + h]."""
    _check(heads, "heads", (F32, BF16), (None, None, None))
    T, H, Dp = heads.shape
    _check(out, "out", heads.dtype, (T, None))
    ld_gate = 0
    if gate is not None:
        _check(gate, "gate", heads.dtype, (T, None))
        ld_gate = gate.shape[1]
        if gate_off < 0 or gate_off + (H if per_head else H * vdim) > ld_gate:
            raise KernelError("sigmoid_gate_heads: columns outside the gate")
    if vdim > Dp or out_off < 0 or out_off + H * vdim > out.shape[1]:
        raise KernelError("sigmoid_gate_heads: columns outside the output")
    call("as_sigmoid_gate_heads", _ptr(heads), _DT[heads.dtype], H, vdim, Dp, _ptr(gate), ld_gate, gate_off,
         int(bool(per_head)), float(scale), _ptr(out), out.shape[1], out_off, T, _stream())  # fmt: skip


# ---- mixers with a fixed-size state --------------------------------------------------------------------


def _check_rows(step_rows, num_tokens):
    tok_row, row_first, row_len, row_start, row_slots = step_rows
    _check(row_first, "row_first", I32, (None,))
    R = row_first.shape[0]
    for name, t in (("row_len", row_len), ("row_start", row_start), ("row_slots", row_slots)):
        _check(t, name, I32, (R,))
    if tok_row is not None:
        _check(tok_row, "tok_row", I32, (num_tokens,))
    elif R < num_tokens:
        raise KernelError("tokens that are their own rows need as many rows")
    return R


def _vector_dtype(proj_dtype, *vectors):
    dtypes = {v.dtype for v in vectors if v is not None}
    if len(dtypes) > 1:
        raise KernelError(f"the small tensors of one part come in one dtype, not {sorted(map(str, dtypes))}")
    dtype = dtypes.pop() if dtypes else proj_dtype
    if dtype not in _DT or (proj_dtype == F32 and dtype != F32):
        raise KernelError(f"small tensors in {dtype} do not go with a projection in {proj_dtype}")
    return dtype


CONV_MAX_TAPS = 8


def short_conv(proj, col0, weight, history, step_rows, out, in_bias=None, bias=None, silu=False, writes=True) -> None:
    """Causal convolution per channel over each row's tokens: out[t, c] = act(sum_i weight[c, i] * in[t - (taps-1-i), c]
    + bias[c]) with in = proj[:, col0 + c] + in_bias[c], zeros before a sequence, and before a row the last taps - 1
    inputs of its request from history [slots, taps - 1, C] (fp32), which then moves on by the row (`writes`).
    step_rows: (tok_row or None, row_first, row_len, row_start, row_slots).  out fp32 [T, C]."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    _check(weight, "weight", (F32, BF16), (None, None))
    C, taps = weight.shape
    if not 1 <= taps <= CONV_MAX_TAPS or col0 < 0 or col0 + C > ld:
        raise KernelError(f"short_conv: {taps} taps (1 to {CONV_MAX_TAPS}) or columns {col0}:{col0 + C} of {ld}")
    w_dtype = _vector_dtype(proj.dtype, weight, in_bias, bias)
    for name, b in (("in_bias", in_bias), ("bias", bias)):
        if b is not None:
            _check(b, name, w_dtype, (C,))
    _check(out, "out", F32, (T, C))
    R = _check_rows(step_rows, T)
    _check(history, "history", F32, (None, max(taps - 1, 0), C) if taps > 1 else None)
    tok_row, row_first, row_len, row_start, row_slots = step_rows
    call("as_short_conv", _ptr(proj), _DT[proj.dtype], ld, col0, C, _ptr(in_bias), _ptr(weight), _ptr(bias),
         _DT[w_dtype], taps, int(bool(silu)), _ptr(history), _ptr(tok_row), _ptr(row_first), _ptr(row_len),
         _ptr(row_start), _ptr(row_slots), _ptr(out), T, R, int(bool(writes)), _stream())  # fmt: skip


def delta_prepare(qkv, num_kv_heads, dim, num_heads, proj, b_off, a_off, a_log, dt_bias, beta, decay) -> None:
    """In place on qkv fp32 [T, C] (G query heads, then G key heads, `dim` wide each, then the values): queries and
    keys become unit vectors (x / sqrt(sum x^2 + 1e-6)), the queries also times dim^(-1/2).  beta [T, H] =
    sigmoid(proj[:, b_off + h]); decay [T, H] = exp(-exp(a_log[h]) * softplus(proj[:, a_off + h] + dt_bias[h]))."""
    _check(qkv, "qkv", F32, (None, None))
    T, C = qkv.shape
    G, H = num_kv_heads, num_heads
    _check(proj, "proj", (F32, BF16), (T, None))
    ld = proj.shape[1]
    if C < 2 * G * dim or min(b_off, a_off) < 0 or max(b_off, a_off) + H > ld:
        raise KernelError("delta_prepare: heads outside the convolution's channels or the projection's columns")
    w_dtype = _vector_dtype(proj.dtype, a_log, dt_bias)
    _check(a_log, "a_log", w_dtype, (H,))
    _check(dt_bias, "dt_bias", w_dtype, (H,))
    _check(beta, "beta", F32, (T, H))
    _check(decay, "decay", F32, (T, H))
    call("as_delta_prepare", _ptr(qkv), C, G, dim, H, _ptr(proj), _DT[proj.dtype], ld, b_off, a_off, _ptr(a_log),
         _ptr(dt_bias), _DT[w_dtype], _ptr(beta), _ptr(decay), T, _stream())  # fmt: skip


# Rows of more tokens than this take the delta rule in chunks of 64 (csrc/recurrent.hip, delta_chunks), shorter ones token by
# token: the chunks' two kernels take 25 us for one chunk of 8 to 16 heads of 128 and 4 us for every further one, the scan 0.4 us
# a token (16 heads: 64 tokens 31 against 26 us, 100 tokens 46 and 30, 2,048 tokens 855 and 153; eight rows of 64 46 and 46, of 128
# 83 and 67).  The line lies above one chunk: a step's many rows of up to 64 tokens are the scan's (30 rows of 60 116 and 127).
DELTA_SCAN_MOST = 79
DELTA_CHUNK = 64
DELTA_CHUNK_SCRATCH = 2 * DELTA_CHUNK * DELTA_CHUNK + 3 * DELTA_CHUNK  # floats per chunk and head


def delta_scan(qkv, num_kv_heads, dim, num_heads, vdim, beta, decay, state, step_rows, out, writes=True, slices=0, longest=0) -> None:
    """The gated delta rule over each row's tokens, per head h (keys and queries of head h // (H / G)):
    S <- decay S; u = beta (v - S^T k); S <- S + k u^T; out = S^T q.  state fp32 [slots, H, dim, vdim]; a row
    that starts at position 0 starts from zero.  qkv as `delta_prepare` left it; out fp32 [T, H, vdim].
    slices: into how many lanes a column of the state is cut (1, 2, 4, 8, 16); 0: chosen so that the step's rows,
    heads and column groups fill the GPU (the results differ by the order of the sums only).
    longest: the most tokens that a row brings, if the caller knows it: long rows then run in chunks (heads of 64 or 128
    keys, values in multiples of 16), the short ones of the step beside them as they are."""
    _check(qkv, "qkv", F32, (None, None))
    T, C = qkv.shape
    G, H = num_kv_heads, num_heads
    if H % G or C != 2 * G * dim + H * vdim:
        raise KernelError(f"delta_scan: {C} channels are not 2 x {G} x {dim} + {H} x {vdim}")
    _check(beta, "beta", F32, (T, H))
    _check(decay, "decay", F32, (T, H))
    _check(state, "state", F32, (None, H, dim, vdim))
    _check(out, "out", F32, (T, H, vdim))
    R = _check_rows((None, *step_rows[1:]), 0)
    _, row_first, row_len, row_start, row_slots = step_rows
    chunked = (longest > DELTA_SCAN_MOST and slices == 0 and dim in (64, 128) and vdim % 16 == 0 and C % 4 == 0
               and qkv.data_ptr() % 16 == 0)  # fmt: skip
    args = (_ptr(qkv), C, G, dim, H, vdim, _ptr(beta), _ptr(decay), _ptr(state), _ptr(row_first), _ptr(row_len), _ptr(row_start),
            _ptr(row_slots), int(bool(writes)), _ptr(out), R)  # fmt: skip
    if not chunked or R > 1:
        call("as_delta_scan", *args, int(slices), DELTA_SCAN_MOST if chunked else 0, _stream())
    if chunked:
        chunks = T // DELTA_CHUNK + min(R, T // (DELTA_SCAN_MOST + 1))  # at least as many as the long rows have
        scratch = torch.empty((chunks, H, DELTA_CHUNK_SCRATCH), dtype=F32, device=qkv.device)
        call("as_delta_chunks", *args, DELTA_SCAN_MOST, _ptr(scratch), chunks, _stream())


def delta_finish(o, weight, eps, proj, g_off, act, gate="silu", scale: float = 1.0, out_off: int = 0) -> None:
    """act[t, out_off + h * vdim + j] = scale * o[t, h, j] / rms(o[t, h]) * weight * gate(proj[t, g_off + h * vdim + j]);
    weight [vdim] (shared by the heads) or [H, vdim]; gate "silu" or "sigmoid"; act [T, >= out_off + H * vdim]."""
    _check(o, "o", F32, (None, None, None))
    T, H, vdim = o.shape
    _check(proj, "proj", (F32, BF16), (T, None))
    if g_off < 0 or g_off + H * vdim > proj.shape[1]:
        raise KernelError("delta_finish: the gate lies outside the projection's columns")
    if gate not in ("silu", "sigmoid"):
        raise KernelError(f"delta_finish: a gate is 'silu' or 'sigmoid', not {gate!r}")
    w_dtype = _vector_dtype(proj.dtype, weight)
    per_head = weight.dim() == 2
    _check(weight, "weight", w_dtype, (H, vdim) if per_head else (vdim,))
    _check(act, "act", proj.dtype, (T, None))
    if out_off < 0 or out_off + H * vdim > act.shape[1]:
        raise KernelError("delta_finish: the heads lie outside the output's columns")
    call("as_delta_finish", _ptr(o), H, vdim, _ptr(weight), _DT[w_dtype], int(per_head), float(eps), _ptr(proj),
         _DT[proj.dtype], proj.shape[1], g_off, int(gate == "sigmoid"), float(scale), _ptr(act), act.shape[1], out_off,
         T, _stream())  # fmt: skip


def delta_prepare_channels(qkv, num_kv_heads, dim, num_heads, proj, b_off, steps, a_off, a_log, dt_bias, beta, chan) -> None:
    """As `delta_prepare` for a rule with a decay per head and key channel: chan [T, H, dim] =
    exp(-exp(a_log[h]) * softplus(steps[:, a_off + h * dim + d] + dt_bias[h * dim + d])); a_log [H], dt_bias [H * dim] fp32."""
    _check(qkv, "qkv", F32, (None, None))
    T, C = qkv.shape
    G, H = num_kv_heads, num_heads
    _check(proj, "proj", (F32, BF16), (T, None))
    _check(steps, "steps", proj.dtype, (T, None))
    if C < 2 * G * dim or b_off < 0 or b_off + H > proj.shape[1] or a_off < 0 or a_off + H * dim > steps.shape[1]:
        raise KernelError("delta_prepare_channels: heads outside the convolution's channels or the projections' columns")
    _check(a_log, "a_log", F32, (H,))
    _check(dt_bias, "dt_bias", F32, (H * dim,))
    _check(beta, "beta", F32, (T, H))
    _check(chan, "chan", F32, (T, H, dim))
    call("as_delta_prepare_channels", _ptr(qkv), C, G, dim, H, _ptr(proj), _DT[proj.dtype], proj.shape[1], b_off,
         _ptr(steps), steps.shape[1], a_off, _ptr(a_log), _ptr(dt_bias), _ptr(beta), _ptr(chan), T, _stream())  # fmt: skip


def delta_scan_channels(qkv, num_kv_heads, dim, num_heads, vdim, beta, chan, state, step_rows, out, writes=True, slices=0) -> None:
    """`delta_scan` with a decay per head and key channel, chan fp32 [T, H, dim], acting on the rows of S:
    S <- diag(chan) S; u = beta (v - S^T k); S <- S + k u^T; out = S^T q."""
    _check(qkv, "qkv", F32, (None, None))
    T, C = qkv.shape
    G, H = num_kv_heads, num_heads
    if H % G or C != 2 * G * dim + H * vdim:
        raise KernelError(f"delta_scan_channels: {C} channels are not 2 x {G} x {dim} + {H} x {vdim}")
    _check(beta, "beta", F32, (T, H))
    _check(chan, "chan", F32, (T, H, dim))
    _check(state, "state", F32, (None, H, dim, vdim))
    _check(out, "out", F32, (T, H, vdim))
    R = _check_rows((None, *step_rows[1:]), 0)
    _, row_first, row_len, row_start, row_slots = step_rows
    call("as_delta_scan_channels", _ptr(qkv), C, G, dim, H, vdim, _ptr(beta), _ptr(chan), _ptr(state), _ptr(row_first),
         _ptr(row_len), _ptr(row_start), _ptr(row_slots), int(bool(writes)), _ptr(out), R, int(slices), _stream())  # fmt: skip


MEMORY_MAX_KEY_DIM = 512  # a lane keeps at most 32 rows of a column of the state beside the normaliser's


def memory_prepare(proj, q_off, k_off, v_off, i_off, f_off, num_heads, dim, vdim, i_bias, f_bias, cap, qkv, i_log, f_log) -> None:
    """What a matrix memory's scan reads, in fp32: qkv [T, 2 H dim + H vdim] = the queries times dim^(-1/2), the keys and
    the values out of proj [T, ld]; i_log = cap tanh((proj[:, i_off + h] + i_bias[h]) / cap) and f_log = logsigmoid(cap
    tanh((proj[:, f_off + h] + f_bias[h]) / cap)), both [T, H]."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    H = num_heads
    if min(q_off, k_off, v_off, i_off, f_off) < 0 or max(q_off, k_off) + H * dim > ld or v_off + H * vdim > ld \
            or max(i_off, f_off) + H > ld:  # fmt: skip
        raise KernelError("memory_prepare: columns outside the projection")
    _check(i_bias, "i_bias", F32, (H,))
    _check(f_bias, "f_bias", F32, (H,))
    _check(qkv, "qkv", F32, (T, 2 * H * dim + H * vdim))
    _check(i_log, "i_log", F32, (T, H))
    _check(f_log, "f_log", F32, (T, H))
    call("as_memory_prepare", _ptr(proj), _DT[proj.dtype], ld, q_off, k_off, v_off, i_off, f_off, H, dim, vdim,
         _ptr(i_bias), _ptr(f_bias), float(cap), _ptr(qkv), _ptr(i_log), _ptr(f_log), T, _stream())  # fmt: skip


def memory_scan(qkv, num_heads, dim, vdim, i_log, f_log, state, norm_state, max_state, step_rows, out, writes=True, slices=0) -> None:
    """A matrix memory with exponential gates over each row's tokens, per head, with a running maximum m (0 at a
    sequence's start): m' = max(f + m, i); S' = e^(f + m - m') S + e^(i - m') k v^T; n' likewise with k;
    out = S'^T q / (max(|n' . q|, e^(-m')) + 1e-6).  state [slots, H, dim, vdim], norm_state [slots, H, dim], max_state
    [slots, H], all fp32; qkv, i_log, f_log as `memory_prepare` left them; out fp32 [T, H, vdim]."""
    _check(qkv, "qkv", F32, (None, None))
    T, C = qkv.shape
    H = num_heads
    if C != 2 * H * dim + H * vdim or dim > MEMORY_MAX_KEY_DIM:
        raise KernelError(f"memory_scan: {C} channels are not {H} x (2 x {dim} + {vdim}), or keys wider than {MEMORY_MAX_KEY_DIM}")
    _check(i_log, "i_log", F32, (T, H))
    _check(f_log, "f_log", F32, (T, H))
    _check(state, "state", F32, (None, H, dim, vdim))
    slots = state.shape[0]
    _check(norm_state, "norm_state", F32, (slots, H, dim))
    _check(max_state, "max_state", F32, (slots, H))
    _check(out, "out", F32, (T, H, vdim))
    R = _check_rows((None, *step_rows[1:]), 0)
    _, row_first, row_len, row_start, row_slots = step_rows
    call("as_memory_scan", _ptr(qkv), C, dim, H, vdim, _ptr(i_log), _ptr(f_log), _ptr(state), _ptr(norm_state),
         _ptr(max_state), _ptr(row_first), _ptr(row_len), _ptr(row_start), _ptr(row_slots), int(bool(writes)), _ptr(out),
         R, int(slices), _stream())  # fmt: skip


def rglru_gates(u, ra, ra_bias, ri, ri_bias, lam, c, a_out, x_out) -> None:
    """The two gates of a gated linear recurrence, per block of channels (ra, ri [blocks, bw, bw], out x in):
    r = sigmoid(ra u_b + ra_bias), i = sigmoid(ri u_b + ri_bias); a_out = exp(-c r softplus(lam)),
    x_out = sqrt(1 - a^2) i u.  u, a_out, x_out fp32 [T, width]."""
    _check(u, "u", F32, (None, None))
    T, width = u.shape
    _check(ra, "ra", (F32, BF16), (None, None, None))
    blocks, bw, _ = ra.shape
    if blocks * bw != width or ra.shape[2] != bw:
        raise KernelError(f"rglru_gates: {blocks} blocks of {tuple(ra.shape[1:])} do not make {width} channels")
    _check(ri, "ri", ra.dtype, (blocks, bw, bw))
    for name, v in (("ra_bias", ra_bias), ("ri_bias", ri_bias), ("lam", lam)):
        _check(v, name, ra.dtype)
        if v.numel() != width:
            raise KernelError(f"{name} has {v.numel()} entries for {width} channels")
    _check(a_out, "a_out", F32, (T, width))
    _check(x_out, "x_out", F32, (T, width))
    call("as_rglru_gates", _ptr(u), width, blocks, _ptr(ra), _ptr(ra_bias), _ptr(ri), _ptr(ri_bias), _ptr(lam),
         _DT[ra.dtype], float(c), _ptr(a_out), _ptr(x_out), T, _stream())  # fmt: skip


def rglru_scan(a, x, proj, y_off, y_bias, scale, state, step_rows, out, out_off, writes=True, row_kinds=None) -> None:
    """S = a S + x per channel over each row's tokens (state fp32 [slots, width]; from zero at position 0);
    out[t, out_off + c] = scale * S * gelu_tanh(proj[t, y_off + c] + y_bias[c]).  row_kinds: how many rows bring more than one token and
    how many more than 64, where known (`StepBatch.row_kinds`): how the work is dealt out."""
    _check(a, "a", F32, (None, None))
    T, width = a.shape
    _check(x, "x", F32, (T, width))
    _check(proj, "proj", (F32, BF16), (T, None))
    _check(out, "out", proj.dtype, (T, None))
    if y_off < 0 or y_off + width > proj.shape[1] or out_off < 0 or out_off + width > out.shape[1]:
        raise KernelError("rglru_scan: columns outside the projection or the output")
    w_dtype = _vector_dtype(proj.dtype, y_bias)
    if y_bias is not None:
        _check(y_bias, "y_bias", w_dtype, (width,))
    _check(state, "state", F32, (None, width))
    R = _check_rows((None, *step_rows[1:]), 0)
    _, row_first, row_len, row_start, row_slots = step_rows
    call("as_rglru_scan", _ptr(a), _ptr(x), width, _ptr(proj), _DT[proj.dtype], proj.shape[1], y_off, _ptr(y_bias),
         _DT[w_dtype], float(scale), _ptr(state), _ptr(row_first), _ptr(row_len), _ptr(row_start), _ptr(row_slots),
         int(bool(writes)), _ptr(out), out.shape[1], out_off, R, T, *(row_kinds or (-1, -1)), _stream())  # fmt: skip


# ---- experts ------------------------------------------------------------------------------------------

MOE_TILES = (64, 128)  # pairs of one expert that a tile of the grouped products holds: of few pairs, of many
MOE_MAX_EXPERTS = 1024


MOE_MANY = 32  # pairs an expert from which on tiles of 128 are taken (`moe_tile`)


def _moe_streamed(w, gated: bool) -> bool:
    """Whether the grouped product with w [experts, N_w, K] runs on the kernel that takes its weights straight into registers
    (`as_moe_gemm`: K in whole blocks of 128, outputs in strips of 16, 16-byte rows, 32-bit offsets within an expert)."""
    rows, K = w.shape[1], w.shape[2]
    return (w.dtype == BF16 and K % 128 == 0 and rows % (32 if gated else 16) == 0 and w.data_ptr() % 16 == 0
            and rows * K * 2 <= 0xF0000000)  # fmt: skip


def moe_tile(pairs: int, first, second, gated: bool) -> int:
    """Pairs a tile of a route whose grouped products read `first` [experts, N_w, K] and then `second`; decides speed alone.
    Tiles of 128 come with operands that go straight into LDS, tiles of 64 with weights straight into registers.  The LDS kernel of other
    sizes takes a tile of 128 as two halves, half of whose workgroups then find
    nothing (32 experts of 2,880 at width 2,880, four a token, 1,500 tokens: 892 us in tiles of 64, 973 of 128), and the 32-bit kernel walks
    it in one workgroup (16 experts of 768 at width 1,024, 1,000 tokens of two: 3,944 and 5,852).  Both products of a layer, us in tiles of
    64 / of 128, by pairs an expert (16 experts, two a token where no others are named; gate and up, their values in millions):
                          16        24        38        62        100       162       256
    width 1,024,  25 M    26/25     26/25     27/25     37/28     41/32     56/38     73/48
    1,024 of 1,536, 50 M  37/39     38/35     42/41     51/42     61/47     87/66     112/80
    2,048,        50 M    36/34     37/35     39/36     47/40     70/48     93/61     123/81
    2,048,       101 M    65/64     67/58     71/61     95/65     103/75    153/102   204/133
    4,096,       403 M    217/225   225/229   238/235   341/248   423/303   560/336   791/439
    2,048, 128 experts, 8 a token, 403 M
                          227/228   236/235   255/248   332/264   450/321   596/393   840/505
    (before, weights into registers and pairs through them into LDS: 2,048 and 101 M at 162 pairs 127, 4,096 and 403 M 482).  Inside
    prompts through 8 layers, 4 of them with such experts, us:
                          24            32            38            48            56            64            100           128
    width 1,024,  25 M    1,492/1,495   1,478/1,476   1,517/1,513   1,499/1,496   1,491/1,488   1,503/1,493   1,570/1,567   1,577/1,567
    2,048,       101 M    1,555/1,550   1,560/1,557   1,578/1,544   1,656/1,616   1,735/1,680   1,850/1,762   2,264/2,188   2,467/2,377
    4,096,       403 M    2,693/2,688   2,807/2,773   3,078/3,045   3,250/3,153   3,643/3,418   3,818/3,493   5,151/4,665   5,767/5,172
    From 32 pairs on tiles of 128 lose nowhere; at 20 they lose 6 us at width 4,096."""
    if not (_moe_streamed(first, gated) and _moe_streamed(second, False)):
        return MOE_TILES[0]
    rows = (-(-pairs // MOE_TILES[1]) + first.shape[0]) * MOE_TILES[1]
    if rows * max(first.shape[2], second.shape[2]) * 2 > 0xF0000000:  # the pairs' rows, too, lie at 32-bit offsets there, at 64-bit ones in tiles of 64
        return MOE_TILES[0]
    return MOE_TILES[pairs >= MOE_MANY * first.shape[0]]


def moe_across(pairs: int, experts: int, rows: int) -> int:
    """Weight rows that a workgroup multiplies a tile of 128 pairs with, 256 or, while that leaves half of the compute units idle, 128
    (a tile more for every second expert than the pairs fill).  One product, us of 256 / of 128, 16 experts, two a token: 1,024 rows
    of K = 768, 1,000 tokens 19 14.5, 2,048 tokens 20 26; 1,536 of 1,024, 500 tokens 21 16, 1,000 tokens 23 26; 6,144 of 4,096, 1,500 tokens 217 311."""
    tiles = pairs / MOE_TILES[1] + experts / 2
    return 128 if 2 * tiles * -(-rows // 256) <= compute_units() else 256


class ExpertRoute:
    """Where a step's (token, chosen expert) pairs stand once sorted by expert: what the grouped products read."""

    __slots__ = ("order", "tiles", "counts", "max_tiles", "top", "num_tokens", "pair_weight", "pair_expert", "tile")

    def __init__(self, num_tokens: int, top: int, experts: int, device, tile: int = MOE_TILES[0]):
        pairs, self.tile = num_tokens * top, tile
        self.max_tiles = -(-pairs // self.tile) + experts
        self.order = torch.empty(max(pairs, 1), dtype=I32, device=device)
        self.tiles = torch.empty((self.max_tiles, 3), dtype=I32, device=device)
        self.counts = torch.empty(1, dtype=I32, device=device)
        self.top, self.num_tokens = top, num_tokens
        self.pair_weight = None  # fp32 [pairs]: what each pair weighs, where a router says (else all weigh alike)
        self.pair_expert = None  # int32 [pairs]: each pair's expert, where a router says


def moe_route_table(token_ids, table, experts: int, tile: int = MOE_TILES[0]) -> ExpertRoute:
    """Routes by a table [vocab, top] int32 that names every token id's experts.  tile (here and below): see `moe_tile`."""
    _check(token_ids, "token_ids", I32, (None,))
    _check(table, "table", I32, (None, None))
    vocab, top = table.shape
    if not 1 <= experts <= MOE_MAX_EXPERTS:
        raise KernelError(f"routing sorts up to {MOE_MAX_EXPERTS} experts, not {experts}")
    route = ExpertRoute(token_ids.shape[0], top, experts, token_ids.device, tile)
    call("as_moe_route_table", _ptr(token_ids), _ptr(table), vocab, top, experts, token_ids.shape[0], _ptr(route.order),
         _ptr(route.tiles), _ptr(route.counts), route.max_tiles, 0, route.tile, _stream())  # fmt: skip
    return route


def moe_route_sigmoid(h, router, top: int, tile: int = MOE_TILES[0]) -> ExpertRoute:
    """Routes by a router's scores: z = router h in fp32, s = sigmoid(z), a token's `top` experts those with the
    largest s, weighing s / (their sum + 1e-20).  h [T, K], router [experts, K] of one dtype.  The route carries
    `pair_weight` fp32 [T * top] for `moe_combine`."""
    return moe_route_scores(h, router, top, "sigmoid", tile=tile)


ROUTER_SCORES = {"sigmoid": 0, "softmax_of_chosen": 1, "softmax": 2}


def moe_route_scores(h, router, top: int, score: str, bias=None, groups: int = 1, keep_groups: int = 1,
                     weight_scale: float = 1.0, correction=None, identity: int = 0,
                     tile: int = MOE_TILES[0]) -> ExpertRoute:  # fmt: skip
    """Routes by a router's logits z = router h + bias in fp32 (bias fp32 [experts] or None).  score "sigmoid": the
    `top` largest sigmoid(z), weighing s / (their sum + 1e-20); "softmax_of_chosen": the `top` largest z, weighing the
    softmax over those z alone; "softmax": s = softmax(z) over all experts, the `top` largest among the experts of the
    `keep_groups` best of `groups` equal groups of neighbours (a group scores its largest s), weighing s * weight_scale.
    correction fp32 [experts] ("softmax" without groups): the `top` largest s + correction are chosen, weighing s.
    identity: the router's last so many outputs are experts without matrices; their pairs stand in no tile of the route.
    The route carries `pair_weight` fp32 [T * top] and `pair_expert` int32 [T * top] for `moe_combine`."""
    _check(h, "h", (F32, BF16), (None, None))
    T, K = h.shape
    _check(router, "router", h.dtype, (None, K))
    experts = router.shape[0]
    if correction is not None:
        _check(correction, "correction", F32, (experts,))
        if score != "softmax" or groups != 1:
            raise KernelError("corrected choices belong to the score 'softmax' without groups")
    if not 0 <= identity < experts:
        raise KernelError(f"{identity} of {experts} experts have no matrices")
    if score not in ROUTER_SCORES:
        raise KernelError(f"a router scores by one of {sorted(ROUTER_SCORES)}, not by {score!r}")
    if bias is not None:
        _check(bias, "bias", F32, (experts,))
    if not 1 <= top <= experts <= MOE_MAX_EXPERTS:
        raise KernelError(f"routing chooses up to {MOE_MAX_EXPERTS} experts, not {top} of {experts}")
    if score != "softmax" and (groups, keep_groups, weight_scale) != (1, 1, 1.0):
        raise KernelError("groups of experts and a scale of the weights belong to the score 'softmax'")
    if groups < 1 or experts % groups or not 1 <= keep_groups <= groups or keep_groups * (experts // groups) < top:
        raise KernelError(f"{experts} experts in {groups} groups of which {keep_groups} are kept do not give {top} to choose")
    route = ExpertRoute(T, top, experts - identity, h.device, tile)
    pair_expert = route.pair_expert = torch.empty(max(T * top, 1), dtype=I32, device=h.device)
    route.pair_weight = torch.empty(max(T * top, 1), dtype=F32, device=h.device)
    call("as_moe_route_scores", _ptr(h), _ptr(router), _ptr(bias), ROUTER_SCORES[score], _ptr(correction), int(groups),
         int(keep_groups), float(weight_scale), _DT[h.dtype], K, experts, top, T,
         _ptr(pair_expert), _ptr(route.pair_weight), _stream())  # fmt: skip
    call("as_moe_route_table", 0, _ptr(pair_expert), 0, top, experts - identity, T, _ptr(route.order), _ptr(route.tiles),
         _ptr(route.counts), route.max_tiles, int(identity), route.tile, _stream())  # fmt: skip
    return route


def moe_gemm(a, w, route: ExpertRoute, out, gated: bool, per_token: bool, activation: str = None, limit: float = 0.0) -> None:
    """The product of every pair's input with its expert's matrix, w [experts, N_w, K].  per_token: a [T, K] holds
    a row per token (all of a token's pairs read it), else a row per pair.  gated: N_w = 2 N, out[p] =
    silu(w[e, :N] a) * (w[e, N:] a), or with limit > 0 the gated activation with limits (`clamped_gate`); else
    out[p] = w[e] a, or relu(w[e] a)^2 with activation "relu2".  out [pairs, N]: a's dtype, or fp32."""
    if limit < 0 or (limit and not gated):
        raise KernelError("moe_gemm: a limit (positive) belongs to a gated product")
    _check(a, "a", (F32, BF16), (None, None))
    K = a.shape[1]
    pairs = route.num_tokens * route.top
    if a.shape[0] != (route.num_tokens if per_token else pairs):
        raise KernelError(f"moe_gemm: {a.shape[0]} input rows for {route.num_tokens} tokens of {route.top} experts")
    _check(w, "w", a.dtype, (None, None, K))
    N = w.shape[1] // 2 if gated else w.shape[1]
    if gated and w.shape[1] % 2:
        raise KernelError("moe_gemm: gate and up rows come in equal numbers")
    _check(out, "out", (a.dtype, F32), (pairs, N))
    if activation not in (None, "relu2") or (gated and activation):
        raise KernelError(f"moe_gemm: activation {activation!r} (None, or 'relu2' on a product without a gate)")
    if (gated or activation) and out.dtype != a.dtype:
        raise KernelError("moe_gemm: the activated product's result has the inputs' dtype")
    call("as_moe_gemm", _ptr(a), _DT[a.dtype], route.top if per_token else 1, _ptr(w), N, K,
         2 if activation else int(bool(gated)),
         _ptr(route.order), _ptr(route.tiles), _ptr(route.counts), route.max_tiles, _ptr(out), _DT[out.dtype], float(limit),
         route.tile, moe_across(pairs, w.shape[0], w.shape[1]), _stream())  # fmt: skip


def moe_combine(pair_out, top: int, weight: float, out, pair_weight=None, add=None, same=None, pair_expert=None, experts: int = 0) -> None:
    """out[t] = sum_j weight * pair_weight[t * top + j] * pair_out[t * top + j] + add[t]; pair_out fp32 [T * top, N];
    pair_weight fp32 [T * top] (None: 1); add [T, N] of out's dtype (None: nothing).  same [T, N] (out's dtype) with
    pair_expert int32 [T * top]: a pair whose expert is numbered `experts` or more has same[t] as its output."""
    _check(out, "out", (F32, BF16), (None, None))
    T, N = out.shape
    _check(pair_out, "pair_out", F32, (T * top, N))
    if pair_weight is not None:
        _check(pair_weight, "pair_weight", F32, (max(T * top, 1),))
    if add is not None:
        _check(add, "add", out.dtype, (T, N))
    if same is not None:
        _check(same, "same", out.dtype, (T, N))
        _check(pair_expert, "pair_expert", I32, (max(T * top, 1),))
    call("as_moe_combine", _ptr(pair_out), top, float(weight), N, _ptr(out), _DT[out.dtype], T, _ptr(pair_weight),
         _ptr(add), _ptr(same), _ptr(pair_expert) if same is not None else 0, int(experts), _stream())  # fmt: skip


# ---- what a layer does to the stream around its parts ------------------------------------------------------

NORM_MAX_GROUPS = 256
CLAMPED_GATE_ALPHA = 1.702  # the factor inside the sigmoid of the gated activation with limits


def group_norm(x, weight, eps, groups: int, out, delta=None, rows=None, update_x=True) -> None:
    """out[r] = the RMS norm in `groups` equal parts of x[s] (+ delta[s]), times weight; s = rows[r] or r.  x fp32
    [T, n] (receives the sum if update_x), weight fp32 [n], delta and out in the compute dtype."""
    _check(x, "x", F32, (None, None))
    T, n = x.shape
    _check(weight, "weight", F32, (n,))
    _check(out, "out", (F32, BF16), (None, n))
    if delta is not None:
        _check(delta, "delta", out.dtype, (T, n))
    if rows is not None:
        _check(rows, "rows", I32, (out.shape[0],))
    elif out.shape[0] != T:
        raise KernelError("group_norm: one output row per row of the stream")
    if not 1 <= groups <= NORM_MAX_GROUPS or n % groups:
        raise KernelError(f"group_norm: {n} columns do not divide into {groups} groups (at most {NORM_MAX_GROUPS})")
    call("as_group_norm", _ptr(x), _ptr(delta), _ptr(rows), _ptr(weight), float(eps), groups, _ptr(out), _DT[out.dtype],
         out.shape[0], n, int(bool(update_x)), _stream())  # fmt: skip


def group_norm_shift(x, weight, mu, eps, groups: int, step_rows, state, out, writes=True) -> None:
    """The grouped norm of every token's row and a token shift after it: out[t] = h_t + (h' - h_t) * mu with h' the
    normed row of the token before, zeros at a sequence's first token, and for a row's first token what its request's
    slot in `state` [slots, n] fp32 holds; the slot then receives the row's last normed row (unless `writes` is off)."""
    _check(x, "x", F32, (None, None))
    T, n = x.shape
    _check(weight, "weight", F32, (n,))
    _check(mu, "mu", F32, (n,))
    _check(out, "out", (F32, BF16), (T, n))
    _check(state, "state", F32, (None, n))
    _check_rows(step_rows, T)
    tok_row, row_first, row_len, row_start, row_slots = step_rows
    if not 1 <= groups <= NORM_MAX_GROUPS or n % groups:
        raise KernelError(f"group_norm_shift: {n} columns do not divide into {groups} groups (at most {NORM_MAX_GROUPS})")
    call("as_group_norm_shift", _ptr(x), _ptr(weight), _ptr(mu), float(eps), groups, _ptr(tok_row), _ptr(row_first),
         _ptr(row_len), _ptr(row_start), _ptr(row_slots), _ptr(state), _ptr(out), _DT[out.dtype], T, n,
         int(bool(writes)), _stream())  # fmt: skip


def depth_average(x, delta, kept, coef, n: int) -> None:
    """v = x + delta is kept as kept[n]; x = sum_(j < n) coef[j] kept[j] + coef[n] v.  x fp32 [T, w]; delta [T, w] in
    the compute dtype or None; kept fp32 [slots > n, T, w]; coef fp32 [n + 1]."""
    _check(x, "x", F32, (None, None))
    _check(kept, "kept", F32, (None, *x.shape))
    _check(coef, "coef", F32, (n + 1,))
    if not 0 <= n < kept.shape[0]:
        raise KernelError(f"depth_average: result {n} of {kept.shape[0]} kept")
    dtype = F32
    if delta is not None:
        _check(delta, "delta", (F32, BF16), tuple(x.shape))
        dtype = delta.dtype
    call("as_depth_average", _ptr(x), _ptr(delta), _DT[dtype], _ptr(kept), _ptr(coef), n, x.numel(), _stream())


def clamped_gate(gate_up, out, limit: float) -> None:
    """out = g sigmoid(1.702 g) (u + 1) with g = min(gate, limit), u = clamp(up, -limit, limit); gate_up [T, 2 I]:
    a row's gate values, then its up values."""
    _check(gate_up, "gate_up", (F32, BF16), (None, None))
    T, two_i = gate_up.shape
    if two_i % 2 or not limit > 0:
        raise KernelError("clamped_gate: gate and up come in equal numbers, and the limit is positive")
    _check(out, "out", gate_up.dtype, (T, two_i // 2))
    call("as_clamped_gate", _ptr(gate_up), _ptr(out), _DT[gate_up.dtype], T, two_i // 2, float(limit), CLAMPED_GATE_ALPHA,
         _stream())  # fmt: skip


def gemm_clamped_gate(a, w, out, limit: float, choices=None) -> None:
    """out = clamped_gate(a @ w^T, limit): w [2 I, K] holds the gate rows, then the up rows; out [T, I]."""
    M, K = a.shape
    rows = _rows(w)
    inter = rows.shape[0] // 2
    if a.dtype == BF16 and M and limit > 0 and (_few_rows(M, K, inter, GATED_MAX_K, w=w) or _gated_two_tiles(M, K, w)):
        # few rows: the product that streams the weights applies the activation on its way out
        _check(rows, "w", a.dtype, (2 * inter, K))
        _check(out, "out", a.dtype, (M, inter))
        call("as_gemm_bf16_gated_limited", _ptr(a), _ptr(rows), _wave_ptr(w), _ptr(out), M, inter, K, float(limit),
             CLAMPED_GATE_ALPHA, _stream())  # fmt: skip
        return
    gate_up = torch.empty((M, rows.shape[0]), dtype=a.dtype, device=a.device)
    gemm(a, w, gate_up, choices)
    clamped_gate(gate_up, out, limit)


# ---- linear attention with a fixed decay per head -------------------------------------------------------------

ACTIVATIONS = {None: 0, "silu": 1, "sigmoid": 2}
DECAY_SCAN_MAX_DIM = 512


def decay_scan(proj, q_off, k_off, v_off, num_heads, dim, vdim, activation, k_scale, decay, state, step_rows, out,
               writes=True) -> None:  # fmt: skip
    """S = decay_h S + k v^T, o = S^T q per head and token, in the order of a row's tokens.  q, k [heads, dim] and v
    [heads, vdim] are columns q_off.., k_off.., v_off.. of proj [T, ld] after `activation` (None or "silu"), k also
    times k_scale.  decay fp32 [heads]; state fp32 [slots, heads, dim, vdim]; out fp32 [T, heads, vdim]."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    H, D, E = num_heads, dim, vdim
    if activation not in (None, "silu"):
        raise KernelError(f"decay_scan: activation {activation!r} (None or 'silu')")
    if min(H, D, E) < 1 or D > DECAY_SCAN_MAX_DIM or max(q_off + H * D, k_off + H * D, v_off + H * E) > ld or min(q_off, k_off, v_off) < 0:
        raise KernelError(f"decay_scan: {H} heads of {D} and {E} at columns {q_off}, {k_off}, {v_off} of {ld}")
    _check(decay, "decay", F32, (H,))
    _check(state, "state", F32, (None, H, D, E))
    _check(out, "out", F32, (T, H, E))
    R = _check_rows(step_rows, T)
    _, row_first, row_len, row_start, row_slots = step_rows
    call("as_decay_scan", _ptr(proj), _DT[proj.dtype], ld, q_off, k_off, v_off, H, D, E, ACTIVATIONS[activation],
         float(k_scale), _ptr(decay), _ptr(state), _ptr(row_first), _ptr(row_len), _ptr(row_start), _ptr(row_slots), R,
         _ptr(out), int(bool(writes)), _stream())  # fmt: skip


DECAY_CHUNKS_MAX_DIM = 128


def decay_chunks(proj, q_off, k_off, v_off, num_heads, dim, vdim, activation, k_scale, decay, state, step_rows, out,
                 writes=True) -> None:  # fmt: skip
    """What `decay_scan` computes, a row's tokens 32 at a time as fp32 products on the matrix cores: with S the state
    before a chunk of n tokens, o_t = decay^(t+1) S^T q_t + sum_(j <= t) decay^(t-j) (q_t . k_j) v_j and the state
    after it decay^n S + sum_j decay^(n-1-j) k_j v_j^T.  Keys of up to DECAY_CHUNKS_MAX_DIM coordinates."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    H, D, E = num_heads, dim, vdim
    if activation not in (None, "silu"):
        raise KernelError(f"decay_chunks: activation {activation!r} (None or 'silu')")
    if min(H, D, E) < 1 or D > DECAY_CHUNKS_MAX_DIM or max(q_off + H * D, k_off + H * D, v_off + H * E) > ld or min(q_off, k_off, v_off) < 0:
        raise KernelError(f"decay_chunks: {H} heads of {D} and {E} at columns {q_off}, {k_off}, {v_off} of {ld}")
    _check(decay, "decay", F32, (H,))
    _check(state, "state", F32, (None, H, D, E))
    _check(out, "out", F32, (T, H, E))
    R = _check_rows(step_rows, T)
    _, row_first, row_len, row_start, row_slots = step_rows
    call("as_decay_chunks", _ptr(proj), _DT[proj.dtype], ld, q_off, k_off, v_off, H, D, E, ACTIVATIONS[activation],
         float(k_scale), _ptr(decay), _ptr(state), _ptr(row_first), _ptr(row_len), _ptr(row_start), _ptr(row_slots), R,
         _ptr(out), int(bool(writes)), _stream())  # fmt: skip


def decay_step(proj, q_off, k_off, v_off, num_heads, dim, vdim, activation, k_scale, decay, state, step_rows, out,
               writes=True) -> None:  # fmt: skip
    """What `decay_scan` computes for a step in which every row is ONE token (only each row's first token is taken):
    the state is read and written once, in whole lines.  Keys of up to DECAY_CHUNKS_MAX_DIM, values a multiple of 4."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    H, D, E = num_heads, dim, vdim
    if activation not in (None, "silu"):
        raise KernelError(f"decay_step: activation {activation!r} (None or 'silu')")
    if min(H, D, E) < 1 or D > DECAY_CHUNKS_MAX_DIM or E % 4 or max(q_off + H * D, k_off + H * D, v_off + H * E) > ld or min(q_off, k_off, v_off) < 0:
        raise KernelError(f"decay_step: {H} heads of {D} and {E} at columns {q_off}, {k_off}, {v_off} of {ld}")
    _check(decay, "decay", F32, (H,))
    _check(state, "state", F32, (None, H, D, E))
    _check(out, "out", F32, (T, H, E))
    R = _check_rows(step_rows, T)
    _, row_first, row_len, row_start, row_slots = step_rows
    call("as_decay_step", _ptr(proj), _DT[proj.dtype], ld, q_off, k_off, v_off, H, D, E, ACTIVATIONS[activation],
         float(k_scale), _ptr(decay), _ptr(state), _ptr(row_first), _ptr(row_start), _ptr(row_slots), R, _ptr(out),
         int(bool(writes)), _stream())  # fmt: skip


def decay_attention(proj, q_off, k_off, v_off, num_heads, dim, vdim, activation, k_scale, decay, state, step_rows, out,
                    writes=True) -> None:  # fmt: skip
    """What `decay_scan` computes, by whichever kernel suits the step: token by token where every row is one token (a
    decode step: step_rows names no row per token; values in fours through the kernel that moves whole lines) or the keys
    are wider than the chunked kernel takes, else in chunks."""
    if dim > DECAY_CHUNKS_MAX_DIM:
        kernel = decay_scan
    elif step_rows[0] is None:
        kernel = decay_step if vdim % 4 == 0 else decay_scan
    else:
        kernel = decay_chunks
    kernel(proj, q_off, k_off, v_off, num_heads, dim, vdim, activation, k_scale, decay, state, step_rows, out, writes)


# ---- and with a decay per token, head and key channel ------------------------------------------------------------

CHANNEL_RANK_MAX = 960  # widest first step of the decays' two-step projection (a tile of tokens' fills a workgroup's LDS)


def channel_decays(proj, low_off, rank, up, bias, tau, alpha) -> None:
    """alpha[t, c] = sigmoid(z)^(1 / tau), z = up[c] . proj[t, low_off:low_off + rank] + bias[c] in fp32 (never below 1e-9).
    up [C, rank] of proj's dtype, bias fp32 [C], alpha fp32 [T, C]."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    _check(up, "up", proj.dtype, (None, rank))
    C = up.shape[0]
    _check(bias, "bias", F32, (C,))
    _check(alpha, "alpha", F32, (T, C))
    if low_off < 0 or low_off + rank > ld or not 1 <= rank <= CHANNEL_RANK_MAX or not tau > 0:
        raise KernelError(f"channel_decays: {rank} columns at {low_off} of {ld} (at most {CHANNEL_RANK_MAX}), tau {tau}")
    call("as_channel_decays", _ptr(proj), _DT[proj.dtype], ld, low_off, rank, _ptr(up), _ptr(bias), float(tau), _ptr(alpha), C, T,
         _stream())  # fmt: skip


CHANNEL_KERNELS = ("scan", "step", "chunks")


def channel_attention(proj, q_off, k_off, v_off, num_heads, dim, vdim, k_scale, alpha, state, step_rows, out, writes=True,
                      kernel: str = None) -> None:  # fmt: skip
    """S = diag(alpha_t) S + k v^T, o = S^T q per head and token, in the order of a row's tokens.  q, k [heads, dim] and v
    [heads, vdim] are columns of proj [T, ld], k times k_scale; alpha fp32 [T, heads * dim]; state fp32 [slots, heads, dim,
    vdim]; out fp32 [T, heads, vdim].  kernel: "scan" (token by token, keys of up to DECAY_SCAN_MAX_DIM), "step" (every
    row ONE token, the state moved in whole lines: values in fours) or "chunks" (32 tokens at a time on the matrix cores in
    fp32), the last two for keys of up to DECAY_CHUNKS_MAX_DIM; None: by what the step and the sizes allow."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    H, D, E = num_heads, dim, vdim
    if kernel is None:
        if D > DECAY_CHUNKS_MAX_DIM:
            kernel = "scan"
        elif step_rows[0] is None:
            kernel = "step" if E % 4 == 0 else "scan"
        else:
            kernel = "chunks"
    if kernel not in CHANNEL_KERNELS:
        raise KernelError(f"channel_attention: kernel {kernel!r} (one of {CHANNEL_KERNELS})")
    most = DECAY_SCAN_MAX_DIM if kernel == "scan" else DECAY_CHUNKS_MAX_DIM
    if min(H, D, E) < 1 or D > most or max(q_off + H * D, k_off + H * D, v_off + H * E) > ld or min(q_off, k_off, v_off) < 0 \
            or (kernel == "step" and E % 4):  # fmt: skip
        raise KernelError(f"channel_attention ({kernel}): {H} heads of {D} and {E} at columns {q_off}, {k_off}, {v_off} of {ld}")
    _check(alpha, "alpha", F32, (T, H * D))
    _check(state, "state", F32, (None, H, D, E))
    _check(out, "out", F32, (T, H, E))
    R = _check_rows(step_rows, T)
    _, row_first, row_len, row_start, row_slots = step_rows
    lens = () if kernel == "step" else (_ptr(row_len),)
    call(f"as_channel_{kernel}", _ptr(proj), _DT[proj.dtype], ld, q_off, k_off, v_off, H, D, E, float(k_scale), _ptr(alpha),
         _ptr(state), _ptr(row_first), *lens, _ptr(row_start), _ptr(row_slots), R, _ptr(out), int(bool(writes)), _stream())  # fmt: skip


def decay_finish(o, groups: int, eps, gain, proj, g_off, gate_activation, out) -> None:
    """out = norm(o) * gain * act(gate): o fp32 [T, n] normed in `groups` equal parts (RMS, eps inside the root),
    gain fp32 [n] or None, the gate columns g_off.. of proj [T, ld], act "sigmoid" or "silu"; out [T, n] proj's dtype."""
    _check(o, "o", F32, (None, None))
    T, n = o.shape
    _check(proj, "proj", (F32, BF16), (T, None))
    if gain is not None:
        _check(gain, "gain", F32, (n,))
    _check(out, "out", proj.dtype, (T, n))
    if gate_activation not in ("silu", "sigmoid") or groups < 1 or n % groups or g_off < 0 or g_off + n > proj.shape[1]:
        raise KernelError(f"decay_finish: {groups} groups of {n}, gate {gate_activation!r} at column {g_off}")
    call("as_decay_finish", _ptr(o), n, groups, float(eps), _ptr(gain), _ptr(proj), _DT[proj.dtype], proj.shape[1], g_off,
         ACTIVATIONS[gate_activation], _ptr(out), T, _stream())  # fmt: skip


# ---- a state space per head -----------------------------------------------------------------------------------------

STATE_SPACE_MAX_STATE, STATE_SPACE_CHUNKS_MAX_STATE = 512, 128  # widest state: token by token; in chunks and in decode steps
STATE_SPACE_KERNELS = {"scan": 0, "step": 1, "chunks": 2}
STATE_SPACE_FILL = 2  # workgroups per compute unit up to which long rows are cut into segments
STATE_SPACE_MIN_SEGMENT = 64  # tokens


def _state_space_segments(longest: int, tokens: int, workgroups: int) -> int:
    """Tokens of a segment for rows of up to `longest` tokens out of `tokens`, a row or segment being `workgroups` workgroups (0:
    rows stay whole): segments of all rows together fill the GPU, and short rows beside a long one do not keep it whole (a row
    alone is a chain of chunks); rows of less than two segments are not worth a second pass."""
    fair = -(-tokens * workgroups // (STATE_SPACE_FILL * compute_units()))
    seg = max(STATE_SPACE_MIN_SEGMENT, _up32(fair))
    return seg if longest >= 2 * seg else 0


def state_space(xbc, num_heads, groups, state_dim, vdim, proj, step_off, dt_bias, a_log, skip, state, step_rows, out, writes=True,
                longest: int = 0, kernel: str = None, seg_len: int = None) -> None:  # fmt: skip
    """Per head h and token, in the order of a row's tokens, with dt = softplus(proj[:, step_off + h] + dt_bias[h]):
    S = exp(-exp(a_log[h]) dt) S + dt B x^T,  out = S^T C + skip[h] x.
    xbc fp32 [T, heads * vdim + 2 groups * state_dim] laid out [x | B | C], head h reading group h // (heads / groups); proj
    [T, ld] of either type; dt_bias, a_log, skip fp32 [heads]; state fp32 [slots, heads, state_dim, vdim]; out fp32 [T, heads *
    vdim].  kernel: "scan" (token by token, states of up to STATE_SPACE_MAX_STATE), "step" (every row ONE token, the state
    moved in whole lines: values in fours) or "chunks" (32 tokens at a time on the matrix cores in fp32), the last two for
    states of up to STATE_SPACE_CHUNKS_MAX_STATE; None: by what the step and the sizes allow.  longest: the longest row's
    tokens, if the caller knows it: long rows are then cut into segments that run at once; seg_len: tokens of a segment (a
    multiple of 32; 0: rows stay whole), None: chosen here.  Cuts change results by rounding only."""
    _check(xbc, "xbc", F32, (None, None))
    T, channels = xbc.shape
    H, G, N, E = num_heads, groups, state_dim, vdim
    if min(H, G, N, E) < 1 or H % G or channels != H * E + 2 * G * N:
        raise KernelError(f"state_space: {channels} channels are not {H} x {E} + 2 x {G} x {N}, or the heads do not divide")
    _check(proj, "proj", (F32, BF16), (T, None))
    if kernel is None:
        if N > STATE_SPACE_CHUNKS_MAX_STATE:
            kernel = "scan"
        elif step_rows[0] is None:
            kernel = "step" if E % 4 == 0 else "scan"
        else:
            kernel = "chunks"
    if kernel not in STATE_SPACE_KERNELS:
        raise KernelError(f"state_space: kernel {kernel!r} (one of {sorted(STATE_SPACE_KERNELS)})")
    most = STATE_SPACE_MAX_STATE if kernel == "scan" else STATE_SPACE_CHUNKS_MAX_STATE
    if N > most or (kernel == "step" and E % 4) or step_off < 0 or step_off + H > proj.shape[1]:
        raise KernelError(f"state_space ({kernel}): a state of {N} x {E}, steps at column {step_off} of {proj.shape[1]}")
    for name, t in (("dt_bias", dt_bias), ("a_log", a_log), ("skip", skip)):
        _check(t, name, F32, (H,))
    _check(state, "state", F32, (None, H, N, E))
    _check(out, "out", F32, (T, H * E))
    R = _check_rows(step_rows, T)
    _, row_first, row_len, row_start, row_slots = step_rows
    seg_state = seg_decay = None
    segments = 0
    if kernel != "chunks":
        seg_len = 0
    elif seg_len is None:
        seg_len = _state_space_segments(longest, T, G * -(-(H // G) * -(-E // 32) // 4))
    if seg_len:
        if seg_len < 0 or seg_len % 32:
            raise KernelError(f"state_space: segments of {seg_len} tokens (a multiple of 32)")
        segments = T // seg_len + R
        seg_state = torch.empty((segments + 1, H, -(-E // 32), -(-N // 32), 1024), dtype=F32, device=xbc.device)
        seg_decay = torch.empty((segments + 1, H), dtype=F32, device=xbc.device)
    call("as_state_space", _ptr(xbc), channels, H, G, N, E, _ptr(proj), _DT[proj.dtype], proj.shape[1], step_off, _ptr(dt_bias),
         _ptr(a_log), _ptr(skip), _ptr(state), _ptr(row_first), _ptr(row_len), _ptr(row_start), _ptr(row_slots), R, _ptr(out),
         int(bool(writes)), STATE_SPACE_KERNELS[kernel], int(seg_len), segments, _ptr(seg_state), _ptr(seg_decay), _stream())  # fmt: skip


def gated_group_norm(y, groups: int, eps, gain, proj, z_off, out) -> None:
    """v = y * silu(z), y fp32 [T, n], z the columns z_off .. of proj [T, ld]; out = v with every one of `groups` equal parts
    divided by its own root mean square (eps inside the root), times gain fp32 [n]; out [T, n] of proj's dtype."""
    _check(y, "y", F32, (None, None))
    T, n = y.shape
    _check(proj, "proj", (F32, BF16), (T, None))
    _check(gain, "gain", F32, (n,))
    _check(out, "out", proj.dtype, (T, n))
    if groups < 1 or n % groups or z_off < 0 or z_off + n > proj.shape[1]:
        raise KernelError(f"gated_group_norm: {groups} groups of {n}, gate at column {z_off} of {proj.shape[1]}")
    call("as_gated_group_norm", _ptr(y), _ptr(proj), _DT[proj.dtype], proj.shape[1], z_off, _ptr(gain), float(eps), n, groups, _ptr(out),
         T, _stream())  # fmt: skip


# ---- attention through a latent ---------------------------------------------------------------------------------


LATENT_MAX_RANK, LATENT_MAX_HEAD_DIM = 1536, 1024  # what eight tokens' latents, or heads, may fill of a workgroup's LDS


def rows_rms_norm(proj, off, n, gain, eps, out) -> None:
    """out = RMS norm of columns off..off + n of proj [T, ld], times gain fp32 [n]; out [T, n] proj's dtype."""
    _check(proj, "proj", (F32, BF16), (None, None))
    _check(gain, "gain", F32, (n,))
    _check(out, "out", proj.dtype, (proj.shape[0], n))
    if off < 0 or off + n > proj.shape[1]:
        raise KernelError("rows_rms_norm: columns outside the rows")
    call("as_rows_rms_norm", _ptr(proj), _DT[proj.dtype], proj.shape[1], off, n, _ptr(gain), float(eps), _ptr(out),
         proj.shape[0], _stream())  # fmt: skip


def latent_kv_store(proj, off, rank, rot, gain, eps, cos_sin, slots, k_pages, v_pages) -> None:
    """Columns off.. of proj [T, ld]: `rank` of the latent (RMS-normed here, times gain fp32 [rank]) and `rot` of the
    shared key part (turned here by cos_sin [T, rot/2, 2] fp32).  [latent | key part | zeros] goes to the key pages
    [pages, 1, bs, width] at slots[t] (< 0: nowhere), [latent | zeros] to the value pages [pages, 1, width, bs]."""
    _check(proj, "proj", (F32, BF16), (None, None))
    T, ld = proj.shape
    _check(gain, "gain", F32, (rank,))
    _check(slots, "slots", I32, (T,))
    _check(k_pages, "k_pages", proj.dtype, (None, 1, None, None))
    pages, _, bs, width = k_pages.shape
    _check(v_pages, "v_pages", proj.dtype, (pages, 1, width, bs))
    if rot:
        _check(cos_sin, "cos_sin", F32, (T, rot // 2, 2))
    if rank < 1 or rot < 0 or rot % 2 or rank + rot > width or off < 0 or off + rank + rot > ld:
        raise KernelError(f"latent_kv_store: a latent of {rank} and a key part of {rot} in pages of {width}, rows of {ld}")
    call("as_latent_kv_store", _ptr(proj), _DT[proj.dtype], ld, off, rank, rot, _ptr(gain), float(eps), _ptr(cos_sin),
         _ptr(slots), _ptr(k_pages), _ptr(v_pages), bs, width, T, _stream())  # fmt: skip


def latent_q_absorb(q, uk, num_heads, dim, rot, rank, cos_sin, out, uk_t=None, q_off: int = 0) -> None:
    """q: columns q_off .. q_off + heads * (dim + rot) of rows [T, ld], uk [heads * dim, rank]: out[t, h] = [uk_h^T q_h[:dim] | q_h[dim:] turned by
    cos_sin | zeros]; out [T, heads, width].  uk_t [heads, rank, dim]: the same matrices transposed, with which
    bfloat16 prompts multiply on the matrix cores."""
    _check(q, "q", (F32, BF16), (None, None))
    T, ld = q.shape
    if q_off < 0 or q_off + num_heads * (dim + rot) > ld:
        raise KernelError("latent_q_absorb: the queries lie outside the rows")
    _check(uk, "uk", q.dtype, (num_heads * dim, rank))
    if uk_t is not None:
        _check(uk_t, "uk_t", q.dtype, (num_heads, rank, dim))
    _check(out, "out", q.dtype, (T, num_heads, None))
    if rot:
        _check(cos_sin, "cos_sin", F32, (T, rot // 2, 2))
    if rank + rot > out.shape[2] or rot % 2 or dim > LATENT_MAX_HEAD_DIM:
        raise KernelError("latent_q_absorb: the latent and the turned part exceed the output's width, or the heads the kernel's")
    call("as_latent_q_absorb", _ptr(q), ld, q_off, _ptr(uk), _ptr(uk_t), _DT[q.dtype], num_heads, dim, rot, rank, _ptr(cos_sin),
         _ptr(out), out.shape[2], T, _stream())  # fmt: skip


def latent_v_expand(heads, uv_t, rank, gate, g_off, out, uv=None) -> None:
    """heads [T, H, width] (the first `rank` coordinates count), uv_t [H, rank, E]: out[t, h E + e] = (sum_r heads[t, h,
    r] uv_t[h, r, e]) * sigmoid(gate[t, g_off + h E + e]); gate [T, ld] or None (no gate); out [T, H * E].  uv [H * E,
    rank]: the same matrices as a checkpoint holds them, with which bfloat16 prompts multiply on the matrix cores."""
    _check(heads, "heads", (F32, BF16), (None, None, None))
    T, H, width = heads.shape
    _check(uv_t, "uv_t", heads.dtype, (H, rank, None))
    E = uv_t.shape[2]
    if uv is not None:
        _check(uv, "uv", heads.dtype, (H * E, rank))
    _check(out, "out", heads.dtype, (T, H * E))
    ld = 0
    if gate is not None:
        _check(gate, "gate", heads.dtype, (T, None))
        ld = gate.shape[1]
        if g_off < 0 or g_off + H * E > ld:
            raise KernelError("latent_v_expand: the gate's columns lie outside its rows")
    if rank > width or rank > LATENT_MAX_RANK:
        raise KernelError("latent_v_expand: the latent is wider than the heads, or than the kernel takes")
    call("as_latent_v_expand", _ptr(heads), _ptr(uv_t), _ptr(uv), _DT[heads.dtype], H, E, rank, width, _ptr(gate), ld,
         g_off, _ptr(out), T, _stream())  # fmt: skip


WIDE_ATTEND_MAX_WIDTH = 2048


def wide_attend(q, k_pages, v_pages, positions, tok_row, block_tables, out, scale, max_context, window=0, keep_first=0,
                softcap=0.0, sink=False, chunk=0) -> None:  # fmt: skip
    """Causal attention of every token's heads q [T, H, width] over kv heads of any width up to
    WIDE_ATTEND_MAX_WIDTH (k_pages [pages, KV, bs, width], v_pages [pages, KV, width, bs]): for pages wider than the
    paged attention kernels' heads.  positions, tok_row [T] int32 (tok_row None: token t is row t); out like q.
    window, keep_first, softcap, sink, chunk, and out in fp32 for bfloat16 heads: as for `attn_single_query`."""
    _check(q, "q", (F32, BF16), (None, None, None))
    T, H, width = q.shape
    sight = _sight(window, keep_first, chunk, softcap, sink, q, out)
    _check(k_pages, "k_pages", q.dtype, (None, None, None, width))
    pages, KV, bs, _ = k_pages.shape
    _check(v_pages, "v_pages", q.dtype, (pages, KV, width, bs))
    if KV < 1 or H % KV:
        raise KernelError(f"attention: {H} query heads do not divide over {KV} kv heads")
    _check(positions, "positions", I32, (T,))
    if tok_row is not None:
        _check(tok_row, "tok_row", I32, (T,))
    _check(block_tables, "block_tables", I32, (None, None))
    if tok_row is None and block_tables.shape[0] < T:
        raise KernelError(f"attention: {T} tokens that are their own rows need as many block tables")
    if width > WIDE_ATTEND_MAX_WIDTH:
        raise KernelError(f"attention: heads of {width} exceed {WIDE_ATTEND_MAX_WIDTH}")
    if max_context > block_tables.shape[1] * bs:
        raise KernelError("attention: block tables are shorter than the longest context")
    call("as_wide_attend", _ptr(q), _ptr(k_pages), _ptr(v_pages), _DT[q.dtype], _ptr(positions), _ptr(tok_row),
         _ptr(block_tables), block_tables.shape[1], _ptr(out), H, KV, width, bs, float(scale),
         *sight, T, _stream())  # fmt: skip
