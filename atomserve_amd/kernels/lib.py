"""Loads the compiled kernel libraries through ctypes and declares their entry points.

The libraries use the HIP runtime that PyTorch has already loaded into the process,
so that device pointers and streams of torch tensors are valid in them; torch is
therefore imported before the first library.  There is no fallback: a kernel whose
library cannot be built or loaded raises.
"""

import ctypes
import functools
import struct
import threading
from ctypes import byref, c_double, c_float, c_int, c_longlong, c_size_t, c_void_p, cast

import torch  # noqa: F401  (loads libamdhip64 first)

from atomserve_amd.kernels import build

P, I, F = c_void_p, c_int, c_float
_CFuncPtr = ctypes.CDLL(None)._FuncPtr.__base__  # what every C function is that ctypes calls
_FLOAT_BITS = struct.Struct("<I")
_WORDS = (c_void_p, c_int, c_longlong, c_size_t)
LIST_INTEGERS, LIST_FLOATS = 32, 4  # of a call that `csrc/launches.hip` makes (its MOST and FLOATS)

# name -> (library, argument types); every entry point returns an int status.
SIGNATURES = {
    "as_embed_gather": ("elementwise", [P, I, P, P, I, I, I, F, P]),
    "as_logits_finish": ("elementwise", [P, c_longlong, F, F, P]),
    "as_rmsnorm": ("elementwise", [P, P, P, P, I, F, P, I, I, I, I, P]),
    "as_rmsnorm_split": ("elementwise", [P, P, I, I, P, P, I, F, P, I, I, I, I, P]),
    "as_rope_table": ("elementwise", [P, P, P, I, I, P]),
    "as_rope_table_scaled": ("elementwise", [P, P, P, I, I, F, P]),
    "as_qk_norm_rope_store": ("elementwise", [P, I, P, P, I, P, P, P, P, P, I, I, I, I, I, F, I, I, P]),
    "as_silu_mul": ("elementwise", [P, P, I, I, I, P]),
    "as_rmsnorm_multi": ("elementwise", [P, P, P, P, P, P, I, F, P, P, I, I, I, I, P]),
    "as_head_norm_store": ("elementwise", [P, I, I, I, I, I, I, I, I, I, I, P, P, I, F, P, P, P, P, I, I, I, P, I, P]),
    "as_gated_add_norm": ("elementwise", [P, P, P, I, I, I, P, F, P, P, I, F, P, I, I, I, I, P, P, P]),
    "as_relu2": ("elementwise", [P, I, I, I, P, I, I, P]),
    "as_whole_norm_store": ("elementwise", [P, I, I, I, I, I, I, I, I, I, I, P, P, P, P, P, F, P, P, I, P, I, F, P, P, P, P, I, I, I, I, P]),
    "as_post_norm_add": ("sandwich", [P, P, P, I, P, P, P, P, F, P, F, P, F, I, I, P, P, I, I, I, P]),
    "as_layer_norm": ("sandwich", [P, P, P, F, P, P, I, I, I, I, P]),
    "as_token_product": ("sandwich", [P, P, P, P, P, I, I, I, P]),
    "as_token_gate": ("sandwich", [P, P, P, I, P, I, I, P]),
    "as_poly_norm": ("sandwich", [P, I, P, F, P, I, I, P]),
    "as_map_difference": ("sandwich", [P, I, I, I, I, F, F, F, P, I, I, I, I, P]),
    "as_streams_step": ("streams", [P, P, I, I, P, I, P, P, F, P, P, F, P, P, I, P]),
    "as_sigmoid_gate_heads": ("elementwise", [P, I, I, I, I, P, I, I, I, F, P, I, I, I, P]),
    "as_short_conv": ("recurrent", [P, I, I, I, I, P, P, P, I, I, I, P, P, P, P, P, P, P, I, I, I, P]),
    "as_delta_prepare": ("recurrent", [P, I, I, I, I, P, I, I, I, I, P, P, I, P, P, I, P]),
    "as_delta_scan": ("recurrent", [P, I, I, I, I, I, P, P, P, P, P, P, P, I, P, I, I, I, P]),
    "as_delta_chunks": ("recurrent", [P, I, I, I, I, I, P, P, P, P, P, P, P, I, P, I, I, P, I, P]),
    "as_delta_finish": ("recurrent", [P, I, I, P, I, I, F, P, I, I, I, I, F, P, I, I, I, P]),
    "as_delta_scan_channels": ("recurrent", [P, I, I, I, I, I, P, P, P, P, P, P, P, I, P, I, I, P]),
    "as_delta_prepare_channels": ("recurrent", [P, I, I, I, I, P, I, I, I, P, I, I, P, P, P, P, I, P]),
    "as_memory_prepare": ("recurrent", [P, I, I, I, I, I, I, I, I, I, I, P, P, F, P, P, P, I, P]),
    "as_memory_scan": ("recurrent", [P, I, I, I, I, P, P, P, P, P, P, P, P, P, I, P, I, I, P]),
    "as_rglru_gates": ("recurrent", [P, I, I, P, P, P, P, P, I, F, P, P, I, P]),
    "as_rglru_scan": ("recurrent", [P, P, I, P, I, I, I, P, I, F, P, P, P, P, P, I, P, I, I, I, I, I, I, P]),
    "as_moe_route_table": ("moe", [P, P, I, I, I, I, P, P, P, I, I, I, P]),
    "as_moe_gemm": ("moe", [P, I, I, P, I, I, I, P, P, P, I, P, I, F, I, I, P]),
    "as_moe_combine": ("moe", [P, I, F, I, P, I, I, P, P, P, P, I, P]),
    "as_moe_route_scores": ("moe", [P, P, P, I, P, I, I, F, I, I, I, I, I, P, P, P]),
    "as_group_norm": ("layer_ops", [P, P, P, P, F, I, P, I, I, I, I, P]),
    "as_group_norm_shift": ("layer_ops", [P, P, P, F, I, P, P, P, P, P, P, P, I, I, I, I, P]),
    "as_depth_average": ("layer_ops", [P, P, I, P, P, I, c_longlong, P]),
    "as_clamped_gate": ("layer_ops", [P, P, I, I, I, F, F, P]),
    "as_decay_scan": ("linear_attention", [P, I, I, I, I, I, I, I, I, I, F, P, P, P, P, P, P, I, P, I, P]),
    "as_decay_chunks": ("linear_attention", [P, I, I, I, I, I, I, I, I, I, F, P, P, P, P, P, P, I, P, I, P]),
    "as_decay_step": ("linear_attention", [P, I, I, I, I, I, I, I, I, I, F, P, P, P, P, P, I, P, I, P]),
    "as_channel_scan": ("linear_attention", [P, I, I, I, I, I, I, I, I, F, P, P, P, P, P, P, I, P, I, P]),
    "as_channel_step": ("linear_attention", [P, I, I, I, I, I, I, I, I, F, P, P, P, P, P, I, P, I, P]),
    "as_channel_chunks": ("linear_attention", [P, I, I, I, I, I, I, I, I, F, P, P, P, P, P, P, I, P, I, P]),
    "as_channel_decays": ("linear_attention", [P, I, I, I, I, P, P, F, P, I, I, P]),
    "as_decay_finish": ("linear_attention", [P, I, I, F, P, P, I, I, I, I, P, I, P]),
    "as_state_space": ("state_space", [P, I, I, I, I, I, P, I, I, I, P, P, P, P, P, P, P, P, I, P, I, I, I, I, P, P, P]),
    "as_gated_group_norm": ("state_space", [P, P, I, I, I, P, F, I, I, P, I, P]),
    "as_rows_rms_norm": ("latent", [P, I, I, I, I, P, F, P, I, P]),
    "as_latent_kv_store": ("latent", [P, I, I, I, I, I, P, F, P, P, P, P, I, I, I, P]),
    "as_latent_q_absorb": ("latent", [P, I, I, P, P, I, I, I, I, I, P, P, I, I, P]),
    "as_latent_v_expand": ("latent", [P, P, P, I, I, I, I, I, P, I, I, P, I, P]),
    "as_wide_attend": ("latent", [P, P, P, I, P, P, P, I, P, I, I, I, I, F, I, I, I, F, I, P, I, I, P]),
    "as_attn_headmix_mfma": ("attention_mix", [P, P, P, P, I, I, I, P, P, P, I, P, P, I, I, I, I, I, F, I, I, I, P, P, P]),
    "as_attn_headmix": ("attention_mix", [P, P, P, I, P, I, I, P, P, P, I, P, P, I, I, I, I, I, F, I, I, P]),
    "as_attn_single_query": ("attention", [P, P, P, I, P, I, P, P, P, I, P, P, P, P, I, I, I, I, F, I, I, I, F, I, P, I, I, I, P]),
    "as_attn_decode_mfma": ("attention", [P, P, P, P, I, P, P, P, I, P, P, P, P, I, I, I, I, F, I, I, I, F, I, P, I, I, I, P]),
    "as_attn_decode_mfma_shared": ("attention", [P, P, P, P, I, P, P, P, I, P, P, P, P, I, I, I, I, F, I, I, I, F, I, P, I, I, I, I, P]),
    "as_attn_decode_fresh": ("attention", [P, P, P, I, P, P, F, I, P, P, P, I, P, P, I, P, P, P, P, I, I, I, I, F, I, I, I, P]),
    "as_attn_prefill_mfma": ("attention", [P, P, P, P, I, P, I, P, I, I, I, I, F, I, I, I, F, I, P, I, I, I, I, P, P, P, P]),
    "as_attn_mixed_mfma": ("attention", [P, P, P, P, I, P, I, P, P, P, I, P, I, I, I, I, F, I, I, I, I, P, P, P, P, P, P, I, I, P]),
    "as_attn_f32": ("attention", [P, P, P, P, I, I, P, I, P, P, P, I, P, P, P, P, I, I, I, I, F, I, I, I, F, I, P, I, I, I, P]),
    "as_attn_f32_fresh": ("attention", [P, P, P, P, P, F, I, P, P, P, I, P, P, I, P, P, P, P, I, I, I, I, F, I, I, I, P]),
    "as_gemm_f32": ("gemm_f32", [P, P, P, I, I, I, I, P]),
    "as_gemm_f32_gated": ("gemm_f32", [P, P, P, I, I, I, I, P]),
    "as_gemm_f32_link": ("gemm_f32", [P, P, P, P, P, P, I, I, I, P]),
    "as_gemm_f32_scaled": ("gemm_f32", [P, P, I, F, P, P, I, I, I, I, P]),
    "as_gemm_f32_split": ("gemm_f32", [P, P, P, I, I, I, I, P]),
    "as_gemm_bf16_skinny": ("gemm", [P, P, P, P, I, I, I, I, I, P]),
    "as_gemm_bf16_gated": ("gemm", [P, P, P, P, I, I, I, P]),
    "as_gemm_bf16_gated_limited": ("gemm", [P, P, P, P, I, I, I, F, F, P]),
    "as_gemm_bf16_link": ("gemm", [P, P, P, P, P, P, P, I, I, I, P]),
    "as_gemm_bf16_scaled": ("gemm", [P, P, I, F, P, P, P, I, I, I, I, P]),
    "as_wave_order": ("gemm", [P, P, I, I, P]),
    "as_gemm_bf16_tile": ("gemm", [P, P, P, P, P, I, I, I, I, I, I, I, P]),
    "as_gemm_bf16_wide": ("gemm_wide", [P, P, P, I, I, I, I, I, I, P]),
    "as_blas_plan": ("blas", [I, I, I, I, c_size_t]),
    "as_blas_candidate_index": ("blas", [I, I, I, I, c_size_t, I]),
    "as_blas_adopt": ("blas", [I, I, I, I, c_size_t, I]),
    "as_blas_prepare_adoption": ("blas", []),
    "as_blas_gemm": ("blas", [P, P, P, I, I, I, I, I, P, c_size_t, P]),
    "as_launch_list": ("launches", [P, c_longlong, P, I, P]),
    "as_argmax": ("sampling", [P, P, I, I, P]),
    "as_sample": ("sampling", [P, I, I, P, P, P, P, P, P, P]),
    "as_sample_split": ("sampling", [P, I, I, P, P, P, P, P, P, P, P, P]),
    "as_apply_penalty": ("sampling", [P, P, P, P, I, I, P]),
    "as_topk": ("sampling", [P, I, I, I, P, P, P]),
}

STATUS = {-1: "unsupported dtype", -2: "unsupported shape or size", -3: "kernel launch failed",
          -4: "partial results exceed the library's static scratch array"}

_libs: dict = {}
_funcs: dict = {}


class KernelError(RuntimeError):
    pass


def _library(name: str):
    if name not in _libs:
        path = build.library_path(name)
        try:
            _libs[name] = ctypes.CDLL(path)
        except OSError as e:
            raise KernelError(f"cannot load {path}: {e}") from e
    return _libs[name]


def entry(name: str):
    """The ctypes function `name`, loading (and if needed compiling) its library."""
    fn = _funcs.get(name)
    if fn is None:
        lib_name, argtypes = SIGNATURES[name]
        try:
            fn = getattr(_library(lib_name), name)
        except AttributeError as e:
            raise KernelError(f"lib_{lib_name}.so has no entry point {name}") from e
        fn.argtypes = argtypes
        fn.restype = c_int
        _funcs[name] = fn
    return fn


class _Watch(threading.local):
    """What this thread writes down: the calls of entry points and the tensors whose addresses they were given."""

    calls = None
    held = None
    spoiled = False  # something ran that is not a call of an entry point, or not the call that the next time would make


watch = _Watch()


def call(name: str, *args) -> None:
    fn = entry(name)
    status = fn(*args)
    if status != 0:
        raise KernelError(f"{name}: {STATUS.get(status, status)}")
    if watch.calls is not None:
        watch.calls.append((name, fn, args))


@functools.lru_cache(maxsize=256)
def _list_places(argtypes: tuple):
    """The arguments of such types that are integers or addresses, those that are 32-bit floats, and the integers' places among their
    like, as `csrc/launches.hip` wants them; None where a list holds no such call."""
    floats = [at for at, kind in enumerate(argtypes) if kind is c_float]
    ints = [at for at, kind in enumerate(argtypes) if kind in _WORDS]
    if len(ints) + len(floats) < len(argtypes) or len(ints) > LIST_INTEGERS or len(floats) > LIST_FLOATS:
        return None
    return ints, floats, {at: i for i, at in enumerate(ints)}


class Launches:
    """The launches that a piece of code makes (`with Launches() as made:`), to be made again with other
    addresses: `made.aim(sources)`, then `made.again(targets)` for as many lists of targets as there are: wherever a
    call was given sources[i], it is given targets[i].  All else in the calls stays: who makes them again answers for it that
    what lies at targets[i] has the type, the shape and the layout of what lies at sources[i].  The tensors that the calls read and wrote are held as long as this
    object lives, so that nobody else is given their memory between two repetitions."""

    def __enter__(self):
        if watch.calls is not None:
            raise KernelError("launches are written down by one list at a time")
        self.calls, self.held = [], []
        watch.calls, watch.held, watch.spoiled = self.calls, self.held, False
        return self

    def __exit__(self, *error):
        self.whole = not watch.spoiled
        watch.calls = watch.held = None
        return False

    def aim(self, sources: list) -> None:
        place = {address: i for i, address in enumerate(sources) if address}
        self.patched = [(name, fn, list(args), [(at, place[v]) for at, v in enumerate(args) if type(v) is int and v in place])
                        for name, fn, args in self.calls]  # fmt: skip
        met = {i for *_, patches in self.patched for _, i in patches}
        # sources with the address of one that the calls were given: which of them it was is not known
        self.same = [(i, place[a]) for i, a in enumerate(sources) if a and place[a] in met and place[a] != i]
        self.met = sorted(met.union(i for i, _ in self.same))
        self.program = self._program()

    def _program(self):
        """The calls as `csrc/launches.hip` takes them: integers and addresses, 32-bit floats, and where targets go; None where one of
        them is not of that kind: an entry point that is no C function, more arguments than a call of a list has or arguments of other types."""
        words = []
        for _, fn, args, patches in self.patched:
            known = _list_places(tuple(fn.argtypes)) if isinstance(fn, _CFuncPtr) else None
            if known is None or len(args) != len(fn.argtypes):
                return None
            ints, floats, place = known
            words += (cast(fn, c_void_p).value, len(ints), len(floats), len(patches))
            words += [0 if args[at] is None else args[at] for at in ints]
            try:
                words += [_FLOAT_BITS.unpack(c_float(args[at]))[0] for at in floats]
            except TypeError:
                return None
            for at, i in patches:
                words += (place[at], i)
        try:
            return (c_longlong * len(words))(*words)
        except TypeError:  # an argument that is no plain number
            return None

    def fits(self, targets: list) -> bool:
        """Whether `targets` (of use: those at the places `met`) can stand for the sources: one address for one address."""
        return all(targets[i] == targets[j] for i, j in self.same)

    def again(self, targets: list) -> None:
        """All calls in one; one by one where a call is none that a list can hold (`_program`)."""
        if self.program is not None:
            failed = c_int(-1)
            status = entry("as_launch_list")(self.program, len(self.program), (c_longlong * len(targets))(*targets), len(targets), byref(failed))
            if status != 0:
                name = self.calls[failed.value][0] if failed.value >= 0 else "as_launch_list"
                raise KernelError(f"{name}: {STATUS.get(status, status)}")
            return
        for name, fn, args, patches in self.patched:
            for at, i in patches:
                args[at] = targets[i]
            status = fn(*args)
            if status != 0:
                raise KernelError(f"{name}: {STATUS.get(status, status)}")


def loaded_libraries() -> list:
    return sorted(_libs)


__all__ = ["KernelError", "Launches", "call", "entry", "loaded_libraries", "c_double"]
