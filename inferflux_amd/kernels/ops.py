"""Python faces of the HIP kernels.

Every function checks on the host that the operands are on the GPU, contiguous, of the
expected type and of shapes that fit what the kernel and its grid assume, and only then
launches on torch's current stream.  Nothing here falls back to another implementation: a
missing library or a refused size raises.
"""
from __future__ import annotations

import ctypes
import functools
import itertools
from typing import Dict, Iterable, Optional, Tuple

import torch

from .. import log
from .device import ARCH, COMPUTE_UNITS, N_XCD
from .library import KernelBuildError, KernelModule, Variant, load_extension, load_module

P = ctypes.c_void_p
I = ctypes.c_int
F = ctypes.c_float
LL = ctypes.c_longlong

DT_F32, DT_BF16 = 0, 1
_DT = {torch.float32: DT_F32, torch.bfloat16: DT_BF16}

ROPE_NONE, ROPE_SPLIT_HALF, ROPE_CONSECUTIVE = 0, 1, 2
ACT_SILU, ACT_GELU_TANH = 0, 1          # gated activations of a feed-forward: act(gate) * up
ACT_CLAMPED_SWISH = 2                   # ... and min(gate, L) sigmoid(1.702 min(gate, L)) (clamp(up, -L, L) + 1), which takes its limit L
ACT_RELU_SQUARED = 3                    # max(x, 0)^2, for a feed-forward without a gate
ACT_NONE = 4                            # the product as it is (of the products of many rows)
PLAIN_ACTS = (ACT_SILU, ACT_GELU_TANH, ACT_RELU_SQUARED)
_PLAIN_EPILOGUE = {ACT_RELU_SQUARED: 4, ACT_GELU_TANH: 5}     # the activations without a gate that the product for few rows has as an epilogue
_GATED_EPILOGUE = {ACT_SILU: 1, ACT_GELU_TANH: 3}    # ... as the epilogue number of the streaming products

# The matrix-core attention module is compiled per head size, when a model with that head size
# first runs; these sizes are compiled ahead by build_all().
MFMA_HEAD_DIMS_PREBUILT = (16, 32, 64, 128)
MFMA_MAX_HEAD_DIM = 128
# The tile kernel's two tilings: 1 = tiles of 64 rows (four waves of 16), which give twice as many workgroups for
# short portions; 2 = tiles of 128 rows, in which every key and value fetched serves twice as many rows.  At head
# size 128 the tall tiles are the kernel of attn_prefill.hip (eight waves of 16 rows, tiles loaded straight into
# LDS), at the other head sizes attn_mfma.hip's with two query tiles per wave.
TILE_QTS = (1, 2)
# (that kernel is written in gfx950's own instructions, loads into LDS of 16 bytes a lane among them; built for anything
# else, the tall tiles of head size 128 are attn_mfma.hip's as well)
DIRECT_TILE_HEAD_DIM = 128 if ARCH == "gfx950" else None


TIME_MIX = (("TIME_MIX", 1),)           # the variant of gla.hip whose read-out comes before the write, with a bonus


class KernelError(RuntimeError):
    pass


def module_variants() -> Iterable[Tuple[str, Variant]]:
    yield ("cache_manager", ())       # host code: the cache's bookkeeping
    yield ("host_calls", ())          # host code: checks, results and calls of every launch
    yield ("core", ())
    yield ("gemm_f32", ())
    yield ("attn_plain", ())
    yield ("sampling", ())
    yield ("gemm_bf16", ())
    yield ("gemm_wide", ())
    yield ("gemm_ring", ())
    yield ("layernorm", ())
    yield ("latent", ())
    yield ("moe", ())
    yield ("ssm", ())
    yield ("gla", ())
    yield ("gla", TIME_MIX)
    yield ("time_mix", ())
    yield ("matrix_memory", ())
    yield ("retention", ())
    yield ("deltas", ())
    yield ("delta", ())
    yield ("hyper", ())
    yield ("rowwise", ())
    yield ("grouped_gemm", ())
    yield ("moe_few", ())
    yield ("moe_f32", ())
    yield ("attn_f32", ())
    yield ("gemm_tiles", ())
    yield ("ceilings", ())            # measurement only: what the memory gives a kernel that just reads
    for d in MFMA_HEAD_DIMS_PREBUILT:
        for qt in TILE_QTS:
            yield _tile_module(d, qt)[:2]
    if DIRECT_TILE_HEAD_DIM is not None:      # (tall tiles with kept first keys, a sink or a gate at that head size)
        yield _tile_module(DIRECT_TILE_HEAD_DIM, 2, direct=False)[:2]
    for dk, dv in WIDE_DIMS_PREBUILT:
        yield ("attn_wide", (("K_DIM", dk), ("V_DIM", dv)))


def _tile_module(head_dim: int, qt: int, direct: bool = True):
    """(module, variant, entry point, the function that says its tile rows) of the tile kernel for a tiling.  ``direct``
    False: not the kernel that loads straight into LDS (it has no kept first keys, sink or gate)."""
    if qt == 2 and head_dim == DIRECT_TILE_HEAD_DIM and direct:
        return "attn_prefill", (("HEAD_DIM", head_dim),), "ifx_attn_prefill", "ifx_attn_prefill_tile_rows"
    return "attn_mfma", (("HEAD_DIM", head_dim), ("TILE_QT", qt)), "ifx_attn_tiles", "ifx_attn_tile_rows"


def _dt(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise KernelError(f"unsupported element type {t.dtype} (float32 or bfloat16)") from None


def _check_in_python(t: torch.Tensor, name: str, shape=None, dtype=None) -> None:
    if not (isinstance(t, torch.Tensor) and t.is_cuda and t.is_contiguous()):
        if not isinstance(t, torch.Tensor):
            raise KernelError(f"{name}: not a tensor")
        if not t.is_cuda:
            raise KernelError(f"{name}: tensor is on {t.device}; the kernels run on the GPU only")
        raise KernelError(f"{name}: tensor is not contiguous")
    if dtype is not None and t.dtype != dtype:
        raise KernelError(f"{name}: element type {t.dtype}, expected {dtype}")
    if shape is not None:
        ts = t.shape
        ok = len(shape) == len(ts)
        if ok:
            for want, got in zip(shape, ts):
                if want is not None and want != got:
                    ok = False
                    break
        if not ok:
            raise KernelError(f"{name}: shape {tuple(ts)}, expected {tuple(shape)}")


def upload(array, device) -> torch.Tensor:
    """The numpy ``array`` on ``device``, by a copy on the current stream that the host does not wait for: from pinned memory of its own,
    which torch's allocator hands out again only after the copy (from ordinary memory ``to`` waits for everything launched before it).  Not in a capture, whose
    replays would copy what that memory holds by then."""
    if torch.device(device).type != "cuda":
        return torch.from_numpy(array).to(device)
    if torch.cuda.is_current_stream_capturing():
        raise KernelError("upload: a captured step's arrays go into buffers that outlive it")
    pageable = torch.from_numpy(array)
    pinned = torch.empty(pageable.shape, dtype=pageable.dtype, pin_memory=True)
    pinned.copy_(pageable)
    return pinned.to(device, non_blocking=True)


def _call_by_ctypes(mod: KernelModule, fname: str, argtypes, *args) -> None:
    rc = mod.fn(fname, argtypes)(*(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args))
    if rc != 0:
        _call_failed(mod, fname, rc)


def _call_failed(mod: KernelModule, fname: str, rc: int) -> None:
    raise KernelError(f"{fname}: {mod.last_error()} (code {rc})")


_WORDS = {P: "p", I: "i", LL: "l", F: "f"}


def _entry(mod: KernelModule, fname: str, argtypes):
    """What the native call keeps of a function: its address and argument types, or None where one of them is no plain word."""
    f = mod.fn(fname, argtypes)
    types = "".join(_WORDS.get(t) or ("a" if issubclass(t, ctypes._Pointer) else "?") for t in argtypes)
    elements = tuple(t._type_ for t, word in zip(argtypes, types) if word == "a")
    found = mod.entries[fname] = _native.entry(ctypes.cast(f, P).value, types, elements)
    return found


def _empty_in_python(shape: Tuple[int, ...], dtype: torch.dtype, like: torch.Tensor) -> torch.Tensor:
    return torch.empty(shape, dtype=dtype, device=like.device)


def _stream_in_python() -> int:
    return torch.cuda.current_stream().cuda_stream


def _host_forms(load):
    """(the native module or None, check, call, empty, stream): what every launch does on the host, from the extension that ``load`` gives.  Where that cannot
    be built (no compiler, no ROCm headers, another processor: hosts without this GPU, where the package is imported for its configuration and plans) the
    Python forms do the same work; the kernels themselves have no other form."""
    try:
        native = load("host_calls")
    except (KernelBuildError, ImportError, OSError) as e:
        log.warn("kernels", f"launches are checked and called in Python, several times slower: {str(e).splitlines()[0]}")
        return None, _check_in_python, _call_by_ctypes, _empty_in_python, _stream_in_python
    native.connect(_check_in_python, _call_by_ctypes, _call_failed, _entry, ctypes.Array)
    return native, native.check, native.call, native.empty, native.stream


_native, _check, _call, empty, _stream = _host_forms(load_extension)      # (see csrc/host_calls.cpp)


# ----------------------------------------------------------------------------------------
def embedding(ids: torch.Tensor, table: torch.Tensor, scale: float = 1.0) -> torch.Tensor:
    """float32 [T, H] rows of ``table`` [V, H] named by int32 ``ids`` [T] (ids are checked by the caller), times ``scale``."""
    _check(ids, "ids", (None,), torch.int32)
    _check(table, "table", (None, None))
    T, H = ids.shape[0], table.shape[1]
    out = empty((T, H), torch.float32, table)
    _call(load_module("core"), "ifx_embedding", (P, P, I, P, I, I, F, P),
          ids, table, _dt(table), out, T, H, float(scale), _stream())
    return out


def embedding_scaled(ids: torch.Tensor, table: torch.Tensor, norm_weight: torch.Tensor, eps: float, scale: float = 1.0):
    """``embedding`` (times ``scale``) for up to 16 tokens that also prepares the RMS norm (weight ``norm_weight`` [H]) which
    reads the stream first: returns (the float32 stream [T, H], that norm's rows up to the factor per row)."""
    _check(ids, "ids", (None,), torch.int32)
    _check(table, "table", (None, None))
    T, H = ids.shape[0], table.shape[1]
    _check(norm_weight, "norm_weight", (H,))
    if T > 16:
        raise KernelError(f"embedding_scaled: {T} rows (at most 16)")
    out = empty((T, H), torch.float32, table)
    rows = empty((T, H), torch.bfloat16, table)
    pieces = empty((-(-H // 4096), 16), torch.float32, table)
    _call(load_module("core"), "ifx_embedding_norm", (P, P, I, P, I, P, P, P, I, I, F, P),
          ids, table, _dt(table), norm_weight, _dt(norm_weight), out, rows,
          pieces, T, H, float(scale), _stream())
    return out, ScaledRows(rows, pieces, H, eps, norm_weight)


def add_rmsnorm(residual: torch.Tensor, delta: Optional[torch.Tensor], weight: torch.Tensor, eps: float,
                out_dtype: torch.dtype, rows: Optional[torch.Tensor] = None, delta_scale: float = 1.0) -> torch.Tensor:
    """``residual`` [T, H] float32 (+= ``delta_scale`` * ``delta`` in place when given and no ``rows``), then RMSNorm.

    With ``rows`` (int32 [R]) only those rows are normalised, into [R, H], and the residual is
    left untouched.  ``delta`` may also be ``SliceSums``, a ``ScaledDelta`` or a ``DeltaSum``.
    """
    _check(residual, "residual", (None, None), torch.float32)
    T, H = residual.shape
    _check(weight, "weight", (H,))
    n_slices = 1
    if isinstance(delta, DeltaSum):
        if delta_scale != 1.0:
            delta = DeltaSum([(delta, delta_scale)])
        if len(delta.terms) == 1 and not _is_vector(delta.terms[0][0]):
            delta, delta_scale = delta.terms[0]
        else:
            return _add_terms_rmsnorm(residual, delta, weight, eps, out_dtype, rows)
    if isinstance(delta, ScaledDelta):             # a delta with its factor
        delta, delta_scale = delta.value, delta_scale * delta.scale
    if isinstance(delta, SliceSums):               # partial sums: the kernel adds them in slice order
        _check(delta.parts, "delta", (None, T, H), torch.float32)
        n_slices, delta = delta.parts.shape[0], delta.parts
    elif delta is not None:
        _check(delta, "delta", (T, H))
    n = T
    if rows is not None:
        _check(rows, "rows", (None,), torch.int32)
        n = rows.shape[0]
    out = empty((n, H), out_dtype, residual)
    _call(load_module("core"), "ifx_add_rmsnorm", (P, P, I, P, I, P, I, P, I, I, F, I, I, LL, F, P),
          residual, delta, _dt(delta) if delta is not None else 0, weight,
          _dt(weight), out, _DT[out_dtype], rows, n, H, float(eps),
          1 if (delta is not None and rows is None) else 0, n_slices, T * H, float(delta_scale), _stream())
    return out


def _is_vector(t) -> bool:
    return isinstance(t, torch.Tensor) and t.dim() == 1


def _term_args(delta: "DeltaSum", T: int, H: int):
    """(number of terms, pointers, dtypes, slices, slice strides, row strides, factors) as the kernels of deltas.hip take them."""
    n = len(delta.terms)
    if n > MAX_DELTA_TERMS:
        raise KernelError(f"{n} additions at once (at most {MAX_DELTA_TERMS})")
    rows = []
    for v, scale in delta.terms:
        if isinstance(v, SliceSums):
            _check(v.parts, "delta", (None, T, H), torch.float32)
            rows.append((v.parts.data_ptr(), DT_F32, v.parts.shape[0], T * H, H, scale))
        else:
            _check(v, "delta", (H,) if _is_vector(v) else (T, H))
            rows.append((v.data_ptr(), _dt(v), 1, 0, 0 if _is_vector(v) else H, scale))
    col = lambda c_type, i: (c_type * max(n, 1))(*[r[i] for r in rows])
    return n, col(P, 0), col(I, 1), col(I, 2), col(LL, 3), col(I, 4), col(F, 5)


MAX_DELTA_TERMS = 6
MAX_DELTA_PIECES = 64          # ... and tensors, vectors and single slices of all of them that the kernels of deltas.hip hold
_TERM_TYPES = (I, ctypes.POINTER(P), ctypes.POINTER(I), ctypes.POINTER(I), ctypes.POINTER(LL), ctypes.POINTER(I), ctypes.POINTER(F))


def _add_terms_rmsnorm(residual, delta: "DeltaSum", weight, eps, out_dtype, rows):
    T, H = residual.shape
    n = T
    delta = delta.in_pieces(MAX_DELTA_PIECES)
    if rows is not None:
        _check(rows, "rows", (None,), torch.int32)
        n = rows.shape[0]
    out = empty((n, H), out_dtype, residual)
    _call(load_module("deltas"), "ifx_add_terms_rmsnorm", (P, *_TERM_TYPES, P, I, P, I, P, I, I, F, I, P),
          residual, *_term_args(delta, T, H), weight, _dt(weight), out, _DT[out_dtype], rows, n, H,
          float(eps), 0 if rows is not None else 1, _stream())
    return out


def join_stream(residual: torch.Tensor, delta, other: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """[T, 2 H] in ``dtype``: the stream ``residual`` [T, H] (float32) plus ``delta`` (anything ``add_rmsnorm`` takes, or None)
    in the first H columns, ``other`` [T, H] (float32) in the rest.  The stream itself is left as it is."""
    _check(residual, "residual", (None, None), torch.float32)
    T, H = residual.shape
    _check(other, "other", (T, H), torch.float32)
    out = empty((T, 2 * H), dtype, residual)
    delta = DeltaSum.of(delta).in_pieces(MAX_DELTA_PIECES)
    _call(load_module("deltas"), "ifx_join_stream", (P, *_TERM_TYPES, P, P, I, I, I, P),
          residual, *_term_args(delta, T, H), other, out, _DT[dtype], T, H, _stream())
    return out


def query_temperature(positions: torch.Tensor, coef: float, every: int) -> torch.Tensor:
    """float32 [T]: 1 + coef ln(floor((p + 1) / every) + 1) of int32 ``positions`` [T]."""
    _check(positions, "positions", (None,), torch.int32)
    out = empty(positions.shape, torch.float32, positions)
    _call(load_module("core"), "ifx_query_temperature", (P, P, I, F, I, P), positions, out, positions.shape[0],
          float(coef), int(every), _stream())
    return out


def slot_table(tensors) -> torch.Tensor:
    """What ``zero_slot`` reads of ``tensors`` (contiguous, [slots, ...]; the caller keeps them): int64 [n, 2]."""
    for t in tensors:
        _check(t, "state")
    rows = [[t.data_ptr(), t.stride(0) * t.element_size()] for t in tensors]
    return torch.tensor(rows, dtype=torch.int64).to(tensors[0].device)


def zero_slot(table: torch.Tensor, slot: int, n_slots: int) -> None:
    """Slot ``slot`` of every tensor of ``table`` (``slot_table``; each of ``n_slots`` slots) to zero, in one launch."""
    _check(table, "table", (None, 2), torch.int64)
    if not 0 <= slot < n_slots:
        raise KernelError(f"zero_slot: slot {slot} of {n_slots}")
    _call(load_module("core"), "ifx_zero_slot", (P, I, LL, P), table, table.shape[0], int(slot), _stream())


def rope_table(positions: torch.Tensor, inv_freq: torch.Tensor, magnitude: float = 1.0):
    """``magnitude`` times cos and sin [T, pairs] of float(position) * inv_freq, computed in float."""
    _check(positions, "positions", (None,), torch.int32)
    _check(inv_freq, "inv_freq", (None,), torch.float32)
    T, n = positions.shape[0], inv_freq.shape[0]
    cs = empty((T, n), torch.float32, positions)
    sn = empty((T, n), torch.float32, positions)
    _call(load_module("core"), "ifx_rope_table", (P, P, P, P, I, I, F, P),
          positions, inv_freq, cs, sn, T, n, float(magnitude), _stream())
    return cs, sn


def rope_append(qkv: torch.Tensor, bias: Optional[torch.Tensor], slots: Optional[torch.Tensor],
                cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], rope_style: int,
                rotary_dim: int, n_heads: int, n_kv_heads: int, head_dim: int,
                k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor], page_size: int,
                v_head_dim: Optional[int] = None, unit_norm_eps: Optional[float] = None, gate_out: Optional[torch.Tensor] = None,
                v_first: Optional[torch.Tensor] = None, v_mix: float = 0.0, v_out: Optional[torch.Tensor] = None,
                qk_norm: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None, extra_cols: int = 0,
                q_mult: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Bias, rotation and cache write of one step's projections; returns q [T, n_heads, head_dim].

    ``qk_norm`` (q weight [head_dim], k weight [head_dim], eps): before the rotation every q and k head becomes
    x / sqrt(mean(x^2) + eps) * weight.  ``extra_cols``: further columns at the end of every row of ``qkv`` that belong
    to another kernel (a gate that is applied elsewhere).  ``q_mult`` float32 [T]: a factor on every query of a row, applied in
    float before the rounding.

    Optionally: ``unit_norm_eps`` divides every q and k head by its root mean square (eps inside the root) after the
    rotation; ``gate_out`` (float32 [T, n_heads]) receives sigmoid(x + bias) of n_heads further columns behind q, k and v
    (a gate per head on the attention's output); ``v_first`` [T, n_kv_heads v_head_dim] is mixed into the values before
    they are cached, v <- (1 - v_mix) v + v_mix v_first; ``v_out`` receives the values as projected, before any mixing.

    ``qkv`` is [T, (n_heads + n_kv_heads) head_dim + n_kv_heads v_head_dim] when the keys and values are
    written (``slots`` int32 [T] = page * page_size + offset; ``v_head_dim`` None: as wide as the keys), or
    [T, n_heads head_dim] with ``n_kv_heads`` = 0 for a mixer that only reads another's cache.  ``cos`` / ``sin``
    are the step's rotation table [T, rotary_dim / 2] (from rope_table).
    """
    T = qkv.shape[0]
    dv = head_dim if v_head_dim is None else int(v_head_dim)
    gate_cols = n_heads if gate_out is not None else 0
    width = (n_heads + n_kv_heads) * head_dim + n_kv_heads * dv + gate_cols + int(extra_cols)
    n_slices = stride = 0
    if isinstance(qkv, SliceSums):                  # partial sums: the kernel adds them in slice order
        _check(qkv.parts, "qkv", (None, T, width), torch.float32)
        n_slices, stride, dtype, qkv = qkv.parts.shape[0], T * width, qkv.dtype, qkv.parts
    else:
        _check(qkv, "qkv", (T, width))
        dtype = qkv.dtype
    if bias is not None:
        _check(bias, "bias", (width,))
    if rope_style != ROPE_NONE:
        _check(cos, "cos", (T, rotary_dim // 2), torch.float32)
        _check(sin, "sin", (T, rotary_dim // 2), torch.float32)
    if slots is not None:
        _check(slots, "slots", (T,), torch.int32)
        _check(k_cache, "k_cache", (None, n_kv_heads, page_size, head_dim), dtype)
        _check(v_cache, "v_cache", (k_cache.shape[0], n_kv_heads, dv, page_size), dtype)
    elif n_kv_heads != 0:
        raise KernelError("rope_append: keys and values given but no slots to write them to")
    if gate_out is not None:
        _check(gate_out, "gate_out", (T, n_heads), torch.float32)
    for t, nm in ((v_first, "v_first"), (v_out, "v_out")):
        if t is not None:
            _check(t, nm, (T, n_kv_heads * dv), dtype)
    qn = kn = None
    if qk_norm is not None:
        qn, kn, pre_eps = qk_norm
        _check(qn, "q norm weight", (head_dim,))
        _check(kn, "k norm weight", (head_dim,), qn.dtype)
    if q_mult is not None:
        _check(q_mult, "q_mult", (T,), torch.float32)
    q = empty((T, n_heads, head_dim), dtype, qkv)
    _call(load_module("core"), "ifx_rope_append",
          (P, I, P, I, P, P, P, I, I, I, I, I, I, I, P, P, P, I, LL, I, I, P, I, F, P, F, P, P, P, I, F, I, P, P),
          qkv, _DT[dtype], bias, _dt(bias) if bias is not None else 0, slots,
          cos if rope_style != ROPE_NONE else None, sin if rope_style != ROPE_NONE else None, rope_style,
          rotary_dim, T, n_heads, n_kv_heads, head_dim, page_size, q, k_cache, v_cache,
          n_slices, stride, dv, gate_cols, gate_out, 1 if unit_norm_eps is not None else 0,
          float(unit_norm_eps or 0.0), v_first, float(v_mix), v_out, qn, kn,
          _dt(qn) if qn is not None else 0, float(pre_eps) if qn is not None else 0.0, int(extra_cols), q_mult, _stream())
    return q


def swiglu(gate_up: torch.Tensor, interleaved: bool = False, act: int = ACT_SILU, limit: float = 0.0) -> torch.Tensor:
    """act(gate) * up [T, I] from [T, 2I] laid out [gate | up] or, interleaved, gate_0, up_0, gate_1, ...; ``act``:
    ACT_SILU (the default), ACT_GELU_TANH, or ACT_CLAMPED_SWISH with its ``limit`` L: g = min(gate, L),
    u = clamp(up, -L, L), g sigmoid(1.702 g) (u + 1)."""
    _check(gate_up, "gate_up", (None, None))
    T, two_i = gate_up.shape
    if two_i % 2:
        raise KernelError("swiglu: odd width")
    out = empty((T, two_i // 2), gate_up.dtype, gate_up)
    _call(load_module("core"), "ifx_swiglu", (P, P, I, I, I, I, I, F, P),
          gate_up, out, _dt(gate_up), T, two_i // 2, 1 if interleaved else 0, int(act), float(limit), _stream())
    return out


def _delta_args(delta, shape, name):
    """(pointer, dtype code, slices, elements between slices) of a tensor or of a product left as ``SliceSums``."""
    if isinstance(delta, ScaledDelta):
        delta = delta.tensor()
    if isinstance(delta, DeltaSum):
        raise KernelError(f"{name}: several additions at once are the RMS norm's to add; form their sum first")
    if isinstance(delta, SliceSums):
        _check(delta.parts, name, (None, *shape), torch.float32)
        return delta.parts.data_ptr(), DT_F32, delta.parts.shape[0], delta.parts[0].numel()
    _check(delta, name, shape)
    return delta.data_ptr(), _dt(delta), 1, 0


def layernorm(x: torch.Tensor, delta, weight: torch.Tensor, eps: float, out_dtype: torch.dtype,
              rows: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Layer norm with a weight and no bias of the rows of ``x`` [T, H] (float32 or bfloat16), in float:
    (x - mean) / sqrt(mean((x - mean)^2) + eps) * weight.  A ``delta`` (a tensor or ``SliceSums``) is added first,
    and written back into ``x`` unless ``rows`` (int32 [R]) picks the rows to normalise."""
    _check(x, "x", (None, None))
    T, H = x.shape
    _check(weight, "weight", (H,))
    if isinstance(delta, DeltaSum):
        delta = delta.tensor(x)
    dp, dd, n_slices, stride = (0, 0, 1, 0) if delta is None else _delta_args(delta, (T, H), "delta")
    n = T
    if rows is not None:
        _check(rows, "rows", (None,), torch.int32)
        n = rows.shape[0]
    out = empty((n, H), out_dtype, x)
    _call(load_module("layernorm"), "ifx_layernorm", (P, I, P, I, I, LL, P, I, P, I, P, I, I, F, P),
          x, _dt(x), dp, dd, n_slices, stride, weight, _dt(weight), out, _DT[out_dtype],
          rows, n, H, float(eps), _stream())
    return out


def add_layernorm(stream: torch.Tensor, delta, weight: torch.Tensor, eps: float,
                  cast_dtype: Optional[torch.dtype] = None) -> Optional[torch.Tensor]:
    """``stream`` [T, H] (float32) += layer norm (weight, no bias) of ``delta`` [T, H] (a tensor or ``SliceSums``), in
    place.  With ``cast_dtype`` the new stream rounded to that type is returned as well (what a sub-block that reads
    the stream itself takes as its input); with float32 that is the stream."""
    _check(stream, "stream", (None, None), torch.float32)
    T, H = stream.shape
    _check(weight, "weight", (H,))
    dp, dd, n_slices, stride = _delta_args(delta, (T, H), "delta")
    cast = empty((T, H), cast_dtype, stream) if cast_dtype not in (None, torch.float32) else None
    _call(load_module("layernorm"), "ifx_add_layernorm", (P, P, I, I, LL, P, I, P, I, I, I, F, P),
          stream, dp, dd, n_slices, stride, weight, _dt(weight), cast,
          _DT[cast_dtype] if cast is not None else 0, T, H, float(eps), _stream())
    return stream if cast_dtype == torch.float32 else cast


def cast_rows(x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """The float32 rows ``x`` rounded to ``dtype`` (bfloat16)."""
    _check(x, "x", None, torch.float32)
    out = empty(x.shape, dtype, x)
    _call(load_module("layernorm"), "ifx_cast_rows", (P, P, I, LL, P), x, out, _DT[dtype], x.numel(), _stream())
    return out


def latent_finish(y, q_norm: Optional[torch.Tensor], kv_norm: Optional[torch.Tensor], eps: float, cos: Optional[torch.Tensor],
                  sin: Optional[torch.Tensor], rot_dims: int, slots: Optional[torch.Tensor], q_rank: int, kv_rank: int,
                  rot_dim: int, k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor], page_size: int,
                  dtype: torch.dtype) -> Optional[torch.Tensor]:
    """What follows the down projections of attention through a latent.  ``y`` [T, >= q_rank + kv_rank + rot_dim] (a
    tensor or ``SliceSums``) holds per row the query latent, the key/value latent and the shared rotated key part (without
    ``slots`` only the query latent is read, and ``kv_norm`` may be None).
    Returns the query latent under its RMS norm (weight ``q_norm``) [T, q_rank] (None when ``q_rank`` is 0); with
    ``slots`` (int32 [T] = page * page_size + offset) the key/value latent under its RMS norm (``kv_norm``) and the
    key part, its first ``rot_dims`` elements turned by the table ``cos`` / ``sin`` [T, rot_dims / 2], go into the
    cache: K rows [latent | key part] (``k_cache`` [pages, 1, page_size, kv_rank + rot_dim]) and V columns
    (``v_cache`` [pages, 1, kv_rank, page_size], or [pages, 1, kv_rank + rot_dim, page_size] for attention kernels that
    want values as wide as keys: the key part is then written there as well)."""
    T, width = y.shape
    if width < q_rank + (kv_rank + rot_dim if slots is not None else 0):
        raise KernelError(f"latent_finish: rows of {width} hold no query latent of {q_rank}, latent of {kv_rank} and key part of {rot_dim}")
    yp, yd, n_slices, stride = _delta_args(y, (T, width), "y")
    if slots is not None:
        _check(kv_norm, "kv_norm", (kv_rank,))
    any_norm = q_norm if kv_norm is None else kv_norm
    if q_rank:
        _check(q_norm, "q_norm", (q_rank,), any_norm.dtype)
    if rot_dims:
        _check(cos, "cos", (T, rot_dims // 2), torch.float32)
        _check(sin, "sin", (T, rot_dims // 2), torch.float32)
    if slots is not None:
        _check(slots, "slots", (T,), torch.int32)
        _check(k_cache, "k_cache", (None, 1, page_size, kv_rank + rot_dim), dtype)
        _check(v_cache, "v_cache", (k_cache.shape[0], 1, None, page_size), dtype)
        if v_cache.shape[2] not in (kv_rank, kv_rank + rot_dim):
            raise KernelError(f"latent_finish: values of {v_cache.shape[2]} rows (the latent's {kv_rank}, or {kv_rank + rot_dim} with the key part)")
    cq = empty((T, q_rank), dtype, any_norm) if q_rank else None
    _call(load_module("latent"), "ifx_latent_finish", (P, I, I, LL, P, P, I, P, P, I, P, P, P, P, I, I, I, I, I, I, F, I, I, P),
          yp, yd, n_slices, stride, q_norm, kv_norm, _dt(any_norm), cos if rot_dims else None,
          sin if rot_dims else None, rot_dims, slots, cq, k_cache if slots is not None else None,
          v_cache if slots is not None else None, _DT[dtype], T, q_rank, kv_rank, rot_dim, page_size, float(eps),
          v_cache.shape[2] if slots is not None else kv_rank, width, _stream())
    return cq


LATENT_QUERY_MAX_RANK = 1536


def latent_query_takes(T: int, dtype: torch.dtype, dim: int, rot_dim: int, kv_rank: int) -> bool:
    """Whether ``latent_query`` takes a step of ``T`` rows."""
    return (dtype == torch.bfloat16 and 0 < T <= HEADWISE_ROWS_MAX and dim % 8 == 0 and (dim + rot_dim) % 8 == 0 and (kv_rank + rot_dim) % 8 == 0
            and kv_rank <= LATENT_QUERY_MAX_RANK)


def _columns(t: torch.Tensor, name: str, T: int, width: int) -> int:
    """How far apart the rows of ``t`` are: [T, width] in bfloat16, whole or columns of wider rows."""
    if not (isinstance(t, torch.Tensor) and t.is_cuda and t.dtype == torch.bfloat16 and t.shape == (T, width) and t.stride(1) == 1 and t.stride(0) >= width):
        raise KernelError(f"{name}: expected bfloat16 rows or columns of rows [{T}, {width}] on the GPU")
    return t.stride(0)


def latent_query(q: torch.Tensor, latent: torch.Tensor, weight: torch.Tensor, n_heads: int, kv_norm: torch.Tensor, eps: float,
                 cos: Optional[torch.Tensor], sin: Optional[torch.Tensor], rot_dims: int, slots: torch.Tensor, rot_dim: int,
                 k_cache: torch.Tensor, v_cache: torch.Tensor, page_size: int) -> torch.Tensor:
    """``headwise`` of the queries ``q`` [T, n_heads * (K + rot_dim)] (a tail of ``rot_dim`` elements behind each head's K) and ``latent_finish``
    of ``latent`` [T, kv_rank + rot_dim] in one launch, for steps of few rows (``latent_query_takes``).  Both in bfloat16, whole rows or columns of
    wider ones (on 16 bytes the queries)."""
    T = q.shape[0]
    _check(weight, "weight", (n_heads, None, None), q.dtype)
    _, N, K = weight.shape
    kv_rank, x_head = kv_norm.shape[0], K + rot_dim
    q_ld, ld = _columns(q, "q", T, n_heads * x_head), _columns(latent, "latent", T, kv_rank + rot_dim)
    if not latent_query_takes(T, q.dtype, K, rot_dim, kv_rank) or q_ld % 8 or q.data_ptr() % 16:
        raise KernelError(f"latent_query: {T} rows (1-{HEADWISE_ROWS_MAX}), {q_ld} apart, of {n_heads} heads of {K} + {rot_dim}, a latent of {kv_rank}")
    _check(kv_norm, "kv_norm", (kv_rank,))
    if rot_dims:
        _check(cos, "cos", (T, rot_dims // 2), torch.float32)
        _check(sin, "sin", (T, rot_dims // 2), torch.float32)
    _check(slots, "slots", (T,), torch.int32)
    _check(k_cache, "k_cache", (None, 1, page_size, kv_rank + rot_dim), q.dtype)
    _check(v_cache, "v_cache", (k_cache.shape[0], 1, None, page_size), q.dtype)
    out = empty((T, n_heads, N + rot_dim), q.dtype, q)
    _call(load_module("latent"), "ifx_latent_query", (P, I, P, I, P, P, I, I, I, I, I, I, P, P, I, P, I, P, P, P, I, I, I, F, I, P),
          q, q_ld, latent, ld, weight, out, T, n_heads, K, N, x_head, rot_dim, cos if rot_dims else None,
          sin if rot_dims else None, rot_dims, kv_norm, _dt(kv_norm), slots, k_cache, v_cache, kv_rank, rot_dim, page_size, float(eps),
          v_cache.shape[2], _stream())
    return out


def linear_normed_takes(x, weight, rank: int) -> bool:
    """Whether ``linear_normed`` takes ``x`` and this weight, a norm over the first ``rank`` columns of whose product follows: a weight whose tiles end where
    those columns do (weights of 2,049 to 3,584 rows have tiles of 10 to 14, which divide few ranks: there the norm keeps its launch), and rows that
    ``linear`` would not send to the ring in slices, whose sums reach the norm in float (928 x 4,096 to the heads' queries at 9 and 16 rows 17.0, 17.1 us,
    joined 14.0, 16.0, but a cached latent's error against 64 bits is 1.65e-3 so and 2.35e-3 through bfloat16)."""
    if not isinstance(weight, LinearWeight) or weight.order is not None or weight.tiled is None or x.dtype != torch.bfloat16:
        return False
    N, K = weight.rows.shape
    return (weight.rows.dtype == torch.bfloat16 and x.shape[0] <= 16 and N % 8 == 0 and 0 < rank <= N and rank % weight.tile_rows == 0
            and _small_m_kernel(x.shape[0], N, K, True) == "skinny" and not ring_takes_few(x, weight, True))


def normed_columns_take(n_rows: int, weight, rank: int) -> bool:
    """Whether ``linear`` takes ``linear_normed``'s ``ScaledRows`` of ``n_rows`` rows with this weight."""
    return (isinstance(weight, LinearWeight) and weight.rows.dtype == torch.bfloat16 and n_rows <= 16 and rank % 8 == 0 and weight.rows.shape[1] == rank
            and _small_m_kernel(n_rows, weight.rows.shape[0], rank, weight.tiled is not None) == "skinny")


def linear_normed(x, weight: LinearWeight, column_scale: torch.Tensor, rank: int, eps: float):
    """x [M <= 16, K] (a tensor or ``ScaledRows``) times ``weight`` [N, K] transposed, times ``column_scale`` [N], as bfloat16 [M, N], and its first
    ``rank`` columns as ``ScaledRows``: the rows of an RMS norm over them (whose weight the scale's first ``rank`` numbers are) up to the factor."""
    N, K = weight.shape
    if (not isinstance(weight, LinearWeight) or weight.order is not None or weight.tiled is None or x.shape[0] > 16 or N % 8 or K % 8 or not 0 < rank <= N
            or rank % weight.tile_rows):
        raise KernelError(f"linear_normed: not for {x.shape[0]} rows times a {tuple(weight.rows.shape)} weight and a norm over {rank} columns")
    x, scale = _scale_args(x)
    M = x.shape[0]
    _check(x, "x", (M, K), torch.bfloat16)
    _check(weight.rows, "weight", (N, K), torch.bfloat16)
    _check(column_scale, "column_scale", (N,))
    y = empty((M, N), torch.bfloat16, x)
    pieces = empty((-(-N // weight.tile_rows), 16), torch.float32, x)
    _call(load_module("gemm_bf16"), "ifx_skinny_gemm", _SKINNY_ARGS,
          x, weight.tiled, 0, DT_F32, M, N, K, 0, 0, 0, 6, weight.tile_rows, 0, *scale, 0, column_scale,
          1 if column_scale.dtype == torch.float32 else 0, y, pieces, 1.0, 0, 0, _stream())
    return y, ScaledRows(y[:, :rank], pieces[:rank // weight.tile_rows], rank, eps, None)


HEADWISE_ROWS_MAX = 16             # rows of a step up to which a thread forms an output element by itself
HEADWISE_GROUPED_MIN_ROWS = 32     # rows of a step from which the per-head products go to the matrix cores


def headwise_takes_splits(T: int, K: int) -> bool:
    """Whether ``headwise`` takes ``SplitRows`` of ``T`` rows (``K`` elements of each head)."""
    return 0 < T <= HEADWISE_ROWS_MAX and K % 8 == 0 and K <= MFMA_MAX_HEAD_DIM


def headwise(x, weight: torch.Tensor, n_heads: int, x_head: int, tail: int = 0,
             cos: Optional[torch.Tensor] = None, sin: Optional[torch.Tensor] = None, rot_dims: int = 0,
             gate: Optional[Tuple[object, int]] = None) -> torch.Tensor:
    """A product per head: out[t, h, :N] = ``weight``[h] x[t, h] with ``weight`` [H, N, K] and head h's input the K
    elements of row t of ``x`` [T, >= H * x_head] from h * x_head on.  The ``tail`` elements that follow a head's K
    inputs are appended to its output, the first ``rot_dims`` of them turned by the table ``cos`` / ``sin``
    [T, rot_dims / 2] in split-half pairs.  ``gate`` = (rows, column): out[t, h, n] is multiplied by the sigmoid of column
    column + h * N + n of ``rows`` [T, ld] (x's type, or ``SliceSums``), in float.  ``x`` may be attention's ``SplitRows`` (without a tail;
    see ``headwise_takes_splits``), which are joined in float.  Returns [T, H, N + tail] in x's type; sums in
    float."""
    splits = x if isinstance(x, SplitRows) else None
    if splits is None:
        _check(x, "x", (None, None))
    T = x.shape[0]
    _check(weight, "weight", (n_heads, None, None), x.dtype)
    _, N, K = weight.shape
    if x_head < K + tail or x.shape[1] < (n_heads - 1) * x_head + K + tail:
        raise KernelError(f"headwise: {n_heads} heads of {K} + {tail} inputs, {x_head} apart, do not fit rows of {x.shape[1]}")
    if rot_dims:
        _check(cos, "cos", (T, rot_dims // 2), torch.float32)
        _check(sin, "sin", (T, rot_dims // 2), torch.float32)
    out = empty((T, n_heads, N + tail), x.dtype, weight)
    gate_args = (0, 0, 0, 0, 0)
    if gate is not None:
        rows, col = gate
        if isinstance(rows, SliceSums):
            _check(rows.parts, "gate", (None, T, None), torch.float32)
            n, _, ld = rows.parts.shape
            gate_args = (rows.parts.data_ptr(), ld, int(col), n, T * ld)
        else:
            _check(rows, "gate", (T, None), x.dtype)
            gate_args = (rows.data_ptr(), rows.shape[1], int(col), 0, 0)
        if col < 0 or col + n_heads * N > gate_args[1]:
            raise KernelError(f"headwise: {n_heads * N} gates from column {col} on do not fit rows of {gate_args[1]}")
    if splits is not None:
        if tail or splits.n_heads != n_heads or splits.width != x_head or not headwise_takes_splits(T, K):
            raise KernelError(f"headwise: splits of {splits.n_heads} heads of {splits.width} where {n_heads} of {x_head} (K={K}, {T} rows) are read")
        _call(load_module("latent"), "ifx_headwise_splits", (P, P, P, I, I, P, P, I, I, I, I, P, I, I, I, LL, P),
              splits.part_o, splits.part_ml, splits.sinks, splits.n_splits, splits.width, weight, out, T, n_heads, K, N, *gate_args, _stream())
        return out
    tail_only = 0
    if x.dtype == torch.bfloat16 and T >= HEADWISE_GROUPED_MIN_ROWS and K % 8 == 0 and x_head % 8 == 0 and x.shape[1] % 8 == 0:
        # many rows: the products on the matrix cores, and of the other kernel only the tails
        _call(load_module("grouped_gemm"), "ifx_headwise_grouped", (P, P, P, I, I, I, I, I, I, I, P, I, I, I, LL, P),
              x, weight, out, T, n_heads, K, N, x.shape[1], x_head, N + tail, *gate_args, _stream())
        if not tail:
            return out
        tail_only = 1
    _call(load_module("latent"), "ifx_headwise", (P, P, P, I, I, I, I, I, I, I, I, P, P, I, I, P, I, I, I, LL, P),
          x, weight, out, _dt(x), T, n_heads, K, N, x.shape[1], x_head, tail,
          cos if rot_dims else None, sin if rot_dims else None, rot_dims, tail_only, *gate_args, _stream())
    return out


ROUTE_FUSED_MAX_ROWS = 16       # rows up to which the router's kernel forms the logits itself


def moe_route(h: torch.Tensor, router, top: int, groups: int = 1, keep_groups: int = 1, group_top: int = 2,
              softmax: bool = False, renormalize: bool = False, scale: float = 1.0, bias: Optional[torch.Tensor] = None,
              choice_bias: Optional[torch.Tensor] = None):
    """The router of a mixture of experts, in float: scores of ``router`` [E, K] (a tensor or a ``LinearWeight``) times the
    rows of ``h`` [T, K] through a sigmoid (or a softmax over the experts), the ``top`` highest among the experts of the best
    ``keep_groups`` of ``groups`` equal groups of neighbours (a group scores the sum of its ``group_top`` highest).  Returns
    (ids int32 [T, top], weights float32 [T, top]): the chosen scores, divided by their sum with ``renormalize``, times
    ``scale``.  ``bias`` float32 [E] is added to the logits before anything else; ``choice_bias`` float32 [E] is added to the
    scores for the choice alone (the weights stay the scores themselves).  Up to ``ROUTE_FUSED_MAX_ROWS`` rows the kernel forms the logits itself; more rows in bfloat16 get them from
    ``linear`` with float32 sums and output."""
    _check(h, "h", (None, None))
    T, K = h.shape
    rows = router.rows if isinstance(router, LinearWeight) else router
    _check(rows, "router", (None, K), h.dtype)
    E = rows.shape[0]
    # (in 32-bit the kernel forms them whatever the rows: a row's sums then never depend on what shares its step)
    z = linear(h, router, out_dtype=torch.float32) if (T > ROUTE_FUSED_MAX_ROWS and h.dtype == torch.bfloat16) else None
    ids = empty((T, top), torch.int32, h)
    weights = empty((T, top), torch.float32, h)
    if bias is not None:
        _check(bias, "bias", (E,), torch.float32)
    if choice_bias is not None:
        _check(choice_bias, "choice_bias", (E,), torch.float32)
    _call(load_module("moe"), "ifx_moe_route", (P, P, I, P, P, P, I, I, I, I, I, I, I, I, I, F, P, P, P),
          h, rows, _dt(h), z, ids, weights, T, K, E, top, groups, keep_groups,
          group_top, 1 if softmax else 0, 1 if renormalize else 0, float(scale), bias, choice_bias, _stream())
    return ids, weights


def pair_gate_up(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """[E, ff, K] gate and up weights (ff a multiple of 16) as one tensor [E, 2 ff, K] whose rows alternate 16 of gate with
    the same 16 of up: a wave of the grouped product then holds a gate tile and its up tile, and the activation is its
    epilogue."""
    E, ff, K = gate.shape
    if ff % 16 or up.shape != gate.shape:
        raise KernelError(f"pair_gate_up: ff={ff} must be a multiple of 16 and both weights alike")
    return torch.stack([gate.view(E, ff // 16, 16, K), up.view(E, ff // 16, 16, K)], dim=2).reshape(E, 2 * ff, K).contiguous()


def moe_experts(h: torch.Tensor, gate: torch.Tensor, up: Optional[torch.Tensor], down: torch.Tensor, ids: torch.Tensor,
                weights: torch.Tensor, act: int = ACT_SILU, limit: float = 0.0, n_identity: int = 0,
                weigh_input: bool = False) -> torch.Tensor:
    """sum_j weights[t, j] * down[e] (act(gate[e] h_t, up[e] h_t)), e = ids[t, j], row by row: every (row, choice)
    streams its expert's weights (``gate`` / ``up`` [E, ff, K], or ``gate`` [E, 2 ff, K] from ``pair_gate_up`` and ``up``
    None; ``down`` [E, N, ff]; all in h's type).  With ``n_identity`` an id from E upwards names an identity expert, whose
    output is the row itself (N = K then).  ``act``: ACT_SILU, ACT_GELU_TANH, or ACT_CLAMPED_SWISH with its ``limit``.  ``weigh_input``: the weights multiply the experts' inputs instead of their
    outputs (in float, on the sums that the activation reads).  Returns [T, N]."""
    _check(h, "h", (None, None))
    T, K = h.shape
    paired = up is None
    _check(gate, "gate", (None, None, K), h.dtype)
    E, ff = gate.shape[0], gate.shape[1] // (2 if paired else 1)
    if not paired:
        _check(up, "up", (E, ff, K), h.dtype)
    _check(down, "down", (E, None, ff), h.dtype)
    N = down.shape[1]
    top = ids.shape[1]
    _check(ids, "ids", (T, top), torch.int32)
    _check(weights, "weights", (T, top), torch.float32)
    if n_identity and N != K:
        raise KernelError(f"moe_experts: identity experts hand back the row itself, so N={N} must equal K={K}")
    mod = load_module("moe")
    a = empty((T, top, ff), h.dtype, h)
    _call(mod, "ifx_moe_gate_up", (P, P, P, P, P, I, I, I, I, I, I, I, I, F, P, P),
          h, gate, up, ids, a, _dt(h), T, K, ff, top, 1 if paired else 0, E,
          int(act), float(limit), weights if weigh_input else None, _stream())
    out = empty((T, N), h.dtype, h)
    _call(mod, "ifx_moe_down", (P, P, P, P, P, I, I, I, I, I, I, P, I, P),
          a, down, ids, weights, out, _dt(h), T, N, ff, top, E, h, 1 if weigh_input else 0, _stream())
    return out


GROUPED_TILE_ITEMS = 128          # items of one expert to a workgroup of the grouped product (TM in csrc/grouped_gemm.hip),
GROUPED_FEW_ITEMS = 64            # ... of weights in tiles where experts have, on average, up to
GROUPED_FEW_MAX_ITEMS = 90        # so many (us by 128 / by 64 at 1,024 x 704 and 88, 125, 175 items 36 / 31, 37 / 35, 41 / 43; at 2,048 x 1,408 and 64 to 73 items
                                  # 155 / 145, 132 / 128 and 264 / 260, 88 to 100 items 161 / 159, 156 / 153 and 292 / 303, 125 items 179 / 187)
GROUPED_MAX_VALUES = 2 ** 30 - 8192          # values of the rows that the product's offsets of 32 bits reach


GROUPED_WAVE_ITEMS = 192          # ... of the product by four large waves,
GROUPED_WAVE_MIN_ITEMS = 225      # which takes experts of so many items on average
GROUPED_WAVE_MIN_ROUNDS = 2.6     # where its tiles take the chip so many times


def grouped_wave_items(n_items: int, n_experts: int, pair_rows: int) -> int:
    """Items to a tile of the product by four large waves where experts with ``pair_rows`` rows of gate and up take it, else 0.  Its tiles of
    256 x 192 are faster by a sixth where all are full, but an expert's last one is half empty on average and so is the last round of the
    chip (90 draws of 14 to 64 experts, 1,024 or 2,048 wide, 704 or 1,408 inner, both products and the order of the items, its time over
    that of tiles of 128 x 128 by eight waves: beyond both lines 0.83 to 0.98, 0.89 in the mean; 100 to 225 items 0.95 to 1.37, fewer
    1.13 to 1.54; fewer rounds 0.85 to 1.28.  20,400 items of 32 experts, 2,048 wide and 1,408 inner: 537 -> 477 us)."""
    tiles = n_items / GROUPED_WAVE_ITEMS + n_experts / 2
    fits = n_items >= GROUPED_WAVE_MIN_ITEMS * n_experts and tiles * -(-pair_rows // 256) >= GROUPED_WAVE_MIN_ROUNDS * COMPUTE_UNITS
    return GROUPED_WAVE_ITEMS if fits else 0


def grouped_items(n_items: int, n_experts: int, pair_rows: int) -> int:
    """Items to a tile where that is not GROUPED_TILE_ITEMS (0)."""
    return GROUPED_FEW_ITEMS if n_items <= GROUPED_FEW_MAX_ITEMS * n_experts else grouped_wave_items(n_items, n_experts, pair_rows)


def grouped_takes(dtype: torch.dtype, K: int, ff: int) -> bool:
    """Whether the grouped matrix-core product takes experts of these sizes."""
    return dtype == torch.bfloat16 and K % 8 == 0 and ff % 16 == 0


class ExpertTiles:
    """The experts' matrices [E, N, K] in the tiled form that the streaming products read (``tile_weights`` with tiles of 16
    rows, N a multiple of 16), instead of their rows: a wave then asks for 1 KB of contiguous memory at a time."""

    __slots__ = ("tiled", "shape")

    def __init__(self, experts: torch.Tensor):
        E, N, K = experts.shape
        if experts.dtype != torch.bfloat16 or N % 16 or K % 8:
            raise KernelError(f"ExpertTiles: {E} experts of {N} x {K} {experts.dtype} (bfloat16, rows a multiple of 16, columns of 8)")
        self.shape = (E, N, K)
        self.tiled = tile_weights(experts.reshape(E * N, K), None, 16)


def _experts(w, nm: str, shape):
    """(shape, address, whether tiled) of the experts' matrices, checked."""
    if isinstance(w, ExpertTiles):
        if any(want is not None and want != have for want, have in zip(shape, w.shape)):
            raise KernelError(f"{nm}: shape {w.shape} where {shape} is expected")
        return w.shape, w.tiled.data_ptr(), 1
    _check(w, nm, shape, torch.bfloat16)
    return tuple(w.shape), w.data_ptr(), 0


def moe_experts_grouped(h: torch.Tensor, gate_up: torch.Tensor, down: torch.Tensor, ids: torch.Tensor,
                        weights: torch.Tensor, act: int = ACT_SILU, limit: float = 0.0, n_identity: int = 0,
                        weigh_input: bool = False, wave_items: int = -1) -> "SliceSums":
    """The same sum for steps of many rows, on the matrix cores: the (row, choice) items are ordered by expert on the
    device and every expert's weights meet tiles of its items (bfloat16; ``gate_up`` from ``pair_gate_up``).  Returns the
    choices' weighted outputs as ``SliceSums`` [top, T, N] (float32), which the kernel that adds them to the stream sums
    in the order of the choices.  ``n_identity``: ids from E up to E + n_identity name identity experts, whose output is
    the row itself (N = K then); ``act``, ``limit`` and ``weigh_input`` as for ``moe_experts``.  ``wave_items`` (both weights as
    ``ExpertTiles``): tiles of so many items, 192 by four large waves, 64 by eight small ones, 0 of 128, -1 chooses."""
    _check(h, "h", (None, None), torch.bfloat16)
    T, K = h.shape
    gu_shape, gu_ptr, gu_tiled = _experts(gate_up, "gate_up", (None, None, K))
    E, ff = gu_shape[0], gu_shape[1] // 2
    down_shape, down_ptr, down_tiled = _experts(down, "down", (E, None, ff))
    N, top = down_shape[1], ids.shape[1]
    _check(ids, "ids", (T, top), torch.int32)
    _check(weights, "weights", (T, top), torch.float32)
    if not grouped_takes(h.dtype, K, ff):
        raise KernelError(f"moe_experts_grouped: K={K} must be a multiple of 8 and ff={ff} of 16")
    mod = load_module("grouped_gemm")
    if n_identity and N != K:
        raise KernelError(f"moe_experts_grouped: identity experts hand back the row itself, so N={N} must equal K={K}")
    n_items = T * top
    n_real, E = E, E + int(n_identity)
    parts = empty((top, T, N), torch.float32, h)
    portion = GROUPED_MAX_VALUES // K
    if T > portion:
        for r in range(0, T, portion):
            parts[:, r:r + portion] = moe_experts_grouped(h[r:r + portion], gate_up, down, ids[r:r + portion], weights[r:r + portion], act,
                                                          limit, n_identity, weigh_input, wave_items).parts
        return SliceSums(parts, torch.bfloat16)
    if wave_items < 0:
        wave_items = grouped_items(n_items, n_real, 2 * ff) if gu_tiled and down_tiled else 0
    tile_items = wave_items or GROUPED_TILE_ITEMS
    max_tiles = -(-n_items // tile_items) + E          # every expert may end on a tile that is not full
    lists = empty((n_items + 3 * max_tiles + 2,), torch.int32, h)
    sorted_, te, ts, tc, nt = (lists[:n_items], lists[n_items:n_items + max_tiles], lists[n_items + max_tiles:n_items + 2 * max_tiles],
                               lists[n_items + 2 * max_tiles:n_items + 3 * max_tiles], lists[n_items + 3 * max_tiles:])
    _call(mod, "ifx_moe_sort", (P, I, I, I, I, P, P, P, P, P, P), ids, n_items, E, n_real, tile_items, sorted_, te,
          ts, tc, nt, _stream())
    a = empty((n_items, ff), torch.bfloat16, h)          # (in the order of ``sorted_``)
    _call(mod, "ifx_moe_gate_up_grouped", (P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, F, P, I, I, P),
          h, gu_ptr, a, sorted_, te, ts, tc,
          nt, max_tiles, T, K, ff, top, n_real, int(act), float(limit),
          weights if weigh_input else None, gu_tiled, wave_items, _stream())
    _call(mod, "ifx_moe_down_grouped", (P, P, P, P, P, P, P, P, P, I, I, I, I, I, I, P, I, I, I, P),
          a, down_ptr, parts, weights, sorted_, te, ts,
          tc, nt, max_tiles, T, N, ff, top, n_real, h, 1 if weigh_input else 0,
          down_tiled, wave_items, _stream())
    return SliceSums(parts, torch.bfloat16)


MOE_F32_TILE_ITEMS = 64          # items of one expert to a workgroup of the 32-bit tiles
MOE_F32_TOGETHER = 4             # ... or to a wave, whose items then share their expert's weights (see csrc/moe_f32.hip)
MOE_F32_TOGETHER_MIN_VALUES = 20_000_000     # k-values times inner columns of all items from which that pays for the items' order, and
MOE_F32_TOGETHER_MAX_ITEMS = 8               # items to an expert up to which it is faster than tiles
MOE_F32_PORTION = 16384          # rows of a launch at most (a grid has up to 65,535 tiles)


def moe_f32_way(n_items: int, n_experts: int, K: int, ff: int) -> int:
    """Items to a tile of the 32-bit experts: 1, each streams its expert's weights for itself, MOE_F32_TOGETHER or MOE_F32_TILE_ITEMS.  us by 1 / 4 / 64, by items to
    an expert: 0.5 to 0.75 94 / 100 / 246 (32 experts of 2,048 x 1,408), 67 / 75 / 133 (64 of 1,024 x 704); 1 43 / 35 / 112 (16 of 1,024 x 1,408), 175 / 149 / 331 (the 32), but 25 /
    31 / 73 of 16 small ones (16 items of 1,024 x 704, 1.2e7); 2 40 / 38 / 89 of those; 6 443 / 213 / 242 (the 64); 8 274 / 114 / 145 (the 16), 1,217 / 425 / 460 (the 32); 12 to
    16 866 / 333 / 245, 555 / 180 / 149, 2,401 / 698 / 467, and 103 / 62 / 73 of 8 experts."""
    if n_items > MOE_F32_TOGETHER_MAX_ITEMS * n_experts:
        return MOE_F32_TILE_ITEMS
    return MOE_F32_TOGETHER if n_items >= n_experts and n_items * K * ff >= MOE_F32_TOGETHER_MIN_VALUES else 1


def moe_experts_f32(h: torch.Tensor, gate: torch.Tensor, up: torch.Tensor, down: torch.Tensor, ids: torch.Tensor, weights: torch.Tensor,
                    act: int = ACT_SILU, limit: float = 0.0, n_identity: int = 0, weigh_input: bool = False,
                    few: Optional[bool] = None, tile_items: int = 0) -> "SliceSums":
    """``moe_experts`` in 32 bits on the matrix cores (``gate`` / ``up`` [E, ff, K], ``down`` [E, N, ff], float32): the choices' weighted
    outputs as ``SliceSums`` [top, T, N].  An element's sum has one order whatever the number of rows; ``few``: each item streams its
    expert's weights for itself, or items are ordered by expert and meet them in tiles of ``tile_items``, 64 or 4 (None and 0 choose)."""
    _check(h, "h", (None, None), torch.float32)
    T, K = h.shape
    _check(gate, "gate", (None, None, K), torch.float32)
    n_real, ff = gate.shape[0], gate.shape[1]
    _check(up, "up", (n_real, ff, K), torch.float32)
    _check(down, "down", (n_real, None, ff), torch.float32)
    N, top, E = down.shape[1], ids.shape[1], n_real + int(n_identity)
    _check(ids, "ids", (T, top), torch.int32)
    _check(weights, "weights", (T, top), torch.float32)
    if n_identity and N != K:
        raise KernelError(f"moe_experts_f32: identity experts hand back the row itself, so N={N} must equal K={K}")
    parts = empty((top, T, N), torch.float32, h)
    portion = max(1, min(MOE_F32_PORTION, (65535 - E) * MOE_F32_TILE_ITEMS // top))
    if T > portion:
        for r in range(0, T, portion):
            parts[:, r:r + portion] = moe_experts_f32(h[r:r + portion], gate, up, down, ids[r:r + portion].contiguous(), weights[r:r + portion].contiguous(),
                                                      act, limit, n_identity, weigh_input, few, tile_items).parts
        return SliceSums(parts, torch.float32)
    n_items = T * top
    tile_items = moe_f32_way(n_items, n_real, K, ff) if few is None else 1 if few else tile_items or MOE_F32_TILE_ITEMS
    lists, max_tiles = (None, None, None, None, None), 0
    if tile_items > 1:
        max_tiles = -(-n_items // tile_items) + E          # every expert may end on a tile that is not full
        ints = empty((n_items + 3 * max_tiles + 2,), torch.int32, h)
        lists = (ints[:n_items], *(ints[n_items + i * max_tiles:n_items + (i + 1) * max_tiles] for i in range(3)), ints[n_items + 3 * max_tiles:])
        _call(load_module("grouped_gemm"), "ifx_moe_sort", (P, I, I, I, I, P, P, P, P, P, P), ids, n_items, E, n_real, tile_items, *lists, _stream())
    a = empty((n_items, ff), torch.float32, h)
    _call(load_module("moe_f32"), "ifx_moe_f32", (P,) * 13 + (I,) * 10 + (F, I, P), h, gate, up, down, ids, weights, a, parts, *lists, max_tiles,
          tile_items, T, K, ff, N, top, n_real, int(n_identity), int(act), float(limit), 1 if weigh_input else 0, _stream())
    return SliceSums(parts, torch.float32)


MOE_FEW_MAX_ROWS = 64          # rows of a step up to which the experts' weights are streamed once for all of them ...
MOE_FEW_MAX_EXPERTS = 256      # ... and experts (identity experts among them) the kernel that chooses takes


def moe_few_takes(dtype: torch.dtype, T: int, K: int, ff: int, n_routed: int, top: int) -> bool:
    """Whether ``moe_few`` takes a step of ``T`` rows (beyond, an expert has rows enough for tiles through LDS)."""
    return grouped_takes(dtype, K, ff) and 0 < T <= MOE_FEW_MAX_ROWS and n_routed <= MOE_FEW_MAX_EXPERTS and top <= 32


def moe_few_choose(h: torch.Tensor, router, top: int, groups: int = 1, keep_groups: int = 1, group_top: int = 2, softmax: bool = False,
                   renormalize: bool = False, scale: float = 1.0, bias: Optional[torch.Tensor] = None,
                   choice_bias: Optional[torch.Tensor] = None, factor: Optional[torch.Tensor] = None):
    """``moe_route`` for up to 64 rows in bfloat16: the router's logits as a product (float32 sums and output) and a launch that
    chooses.  Returns (ids int32 [T, top], weights float32 [T, top]).  ``h`` may be ``ScaledRows``, whose factors are then written to
    ``factor`` [T] (float32)."""
    h, scale_args = _scale_args(h)
    if (factor is None) != (scale_args[0] == 0):
        raise KernelError("moe_few: scaled rows and a place for their factors go together")
    if factor is not None:
        _check(factor, "factor", (h.shape[0],), torch.float32)
    _check(h, "h", (None, None), torch.bfloat16)
    T, K = h.shape
    rows = router.rows if isinstance(router, LinearWeight) else router
    _check(rows, "router", (None, K), torch.bfloat16)
    E = rows.shape[0]
    if not 0 < T <= MOE_FEW_MAX_ROWS or E > MOE_FEW_MAX_EXPERTS or K % 8 or top > 32:
        raise KernelError(f"moe_few: {T} rows (at most {MOE_FEW_MAX_ROWS}), {E} experts (at most {MOE_FEW_MAX_EXPERTS}), K={K} (a multiple of 8), top {top} (at most 32)")
    for t, nm in ((bias, "bias"), (choice_bias, "choice_bias")):
        if t is not None:
            _check(t, nm, (E,), torch.float32)
    mod, stream = load_module("moe_few"), _stream()
    slices = mod.fn("ifx_moe_logit_slices", (I,))(K)
    z = empty((slices, T, E), torch.float32, h)
    _call(mod, "ifx_moe_logits", (P, P, P, I, I, I, P, I, F, F, P, P), h, rows, z, T, K, E, *scale_args,
          factor, stream)
    ids = empty((T, top), torch.int32, h)
    weights = empty((T, top), torch.float32, h)
    _call(mod, "ifx_moe_choose", (P, I, P, P, I, I, I, I, I, I, I, I, F, P, P, P), z, slices, ids, weights,
          T, E, top, groups, keep_groups, group_top, 1 if softmax else 0, 1 if renormalize else 0, float(scale), bias, choice_bias, stream)
    return ids, weights


def moe_few_experts(h: torch.Tensor, gate_up: torch.Tensor, down: torch.Tensor, ids: torch.Tensor, weights: torch.Tensor, act: int = ACT_SILU,
                    limit: float = 0.0, n_identity: int = 0, weigh_input: bool = False, shared=None, shared_limit: float = 0.0,
                    factor: Optional[torch.Tensor] = None) -> "SliceSums":
    """``moe_experts`` for up to 64 rows in bfloat16: two launches that stream every chosen expert's weights once, whatever the
    number of rows that chose it (``gate_up`` from ``pair_gate_up``; both as tensors or ``ExpertTiles``).  Returns the choices' weighted outputs as ``SliceSums`` [top, T, N] like ``moe_experts_grouped``.
    ``shared``: (gate_up, down) of an expert that every row takes, [1, 2 shared_ff, K] and [1, N, shared_ff] in the experts' form
    (with its own ``shared_limit``): its output is the last of [top + 1, T, N].  ``factor`` [T] (float32): h's rows are to be multiplied by it."""
    if factor is not None:
        _check(factor, "factor", (h.shape[0],), torch.float32)
    _check(h, "h", (None, None), torch.bfloat16)
    T, K = h.shape
    gu_shape, gu_ptr, gu_tiled = _experts(gate_up, "gate_up", (None, None, K))
    n_real, ff = gu_shape[0], gu_shape[1] // 2
    down_shape, down_ptr, down_tiled = _experts(down, "down", (n_real, None, ff))
    N, E, top = down_shape[1], n_real + int(n_identity), ids.shape[1]
    _check(ids, "ids", (T, top), torch.int32)
    _check(weights, "weights", (T, top), torch.float32)
    if not moe_few_takes(h.dtype, T, K, ff, E, top):
        raise KernelError(f"moe_few: {T} rows (at most {MOE_FEW_MAX_ROWS}), {E} experts (at most {MOE_FEW_MAX_EXPERTS}), K={K} (a multiple of 8), ff={ff} (of 16)")
    if n_identity and N != K:
        raise KernelError(f"moe_few: identity experts hand back the row itself, so N={N} must equal K={K}")
    mod, stream = load_module("moe_few"), _stream()
    shared_ff = shared_gu = shared_down = 0
    if shared is not None:
        shape, shared_gu, gu_form = _experts(shared[0], "shared gate_up", (1, None, K))
        shared_ff = shape[1] // 2
        _, shared_down, down_form = _experts(shared[1], "shared down", (1, N, shared_ff))
        if shape[1] % 32 or (gu_form, down_form) != (gu_tiled, down_tiled):
            raise KernelError(f"moe_few: a shared expert of {shape[1]} gate and up rows (a multiple of 32), in the experts' form")
    a = empty((T * (top * ff + shared_ff),), torch.bfloat16, h)
    shared_a = a.data_ptr() + 2 * T * top * ff
    _call(mod, "ifx_moe_few_gate_up", (P, P, P, P, I, I, I, I, I, I, I, F, P, I, P, P, I, F, P, P), h, gu_ptr, a, ids,
          T, E, K, ff, top, n_real, int(act), float(limit), weights if weigh_input else None, gu_tiled,
          shared_gu, shared_a, shared_ff, float(shared_limit), factor, stream)
    parts = empty((top + (1 if shared is not None else 0), T, N), torch.float32, h)
    _call(mod, "ifx_moe_few_down", (P, P, P, P, P, I, I, I, I, I, I, P, I, I, P, P, I, P, P), a, down_ptr, parts,
          weights, ids, T, E, N, ff, top, n_real, h, 1 if weigh_input else 0, down_tiled,
          shared_a, shared_down, shared_ff, factor, stream)
    return SliceSums(parts, torch.bfloat16)


def moe_few(h: torch.Tensor, router, gate_up: torch.Tensor, down: torch.Tensor, top: int, groups: int = 1, keep_groups: int = 1,
            group_top: int = 2, softmax: bool = False, renormalize: bool = False, scale: float = 1.0, bias: Optional[torch.Tensor] = None,
            choice_bias: Optional[torch.Tensor] = None, act: int = ACT_SILU, limit: float = 0.0, n_identity: int = 0,
            weigh_input: bool = False) -> "SliceSums":
    """``moe_few_choose`` and ``moe_few_experts``, one after the other."""
    E = router.shape[0] if isinstance(router, torch.Tensor) else router.rows.shape[0]
    if E != gate_up.shape[0] + int(n_identity):
        raise KernelError(f"router: {E} experts where {gate_up.shape[0]} + {n_identity} are expected")
    ids, weights = moe_few_choose(h, router, top, groups, keep_groups, group_top, softmax, renormalize, scale, bias, choice_bias)
    return moe_few_experts(h, gate_up, down, ids, weights, act, limit, n_identity, weigh_input)


# ----------------------------------------------------------------------------------------
def gemm_f32(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
             out_dtype: Optional[torch.dtype] = None, gated: Optional[int] = None, limit: float = 0.0) -> torch.Tensor:
    """x [M, K] (float32 or bfloat16) times float32 ``weight`` [N, K] transposed, true 32-bit math.  ``gated`` (float32 x, no bias): the
    activation of weight rows of gate and up in turn, the result [M, N / 2] (``limit``: ACT_CLAMPED_SWISH's)."""
    _check(x, "x", (None, None))
    M, K = x.shape
    _check(weight, "weight", (None, K), torch.float32)
    N = weight.shape[0]
    if bias is not None:
        _check(bias, "bias", (N,), torch.float32)
    out_dtype = out_dtype or x.dtype
    out = empty((M, N if gated is None else N // 2), out_dtype, x)
    _call(load_module("gemm_f32"), "ifx_gemm_f32", (P, I, P, P, P, I, I, I, I, I, F, P), x, _dt(x), weight, bias,
          out, _DT[out_dtype], M, N, K, -1 if gated is None else int(gated), float(limit), _stream())
    return out


SKINNY_MAX_M = 64
WIDE_MAX_M = 128           # rows the product that shares x through LDS takes at most ...
WIDE_MANY_ROWS_MAX_N = 16384   # ... beyond 64 of them only for weights of up to this many rows (see _small_m_kernel)


def enable_library_gemm_tuning(max_ms_per_shape: int = 300, filename: Optional[str] = None) -> None:
    """Let the library pick, by timing, the fastest of its kernels for every matrix-product shape it
    meets (torch's TunableOp over hipBLASLt and rocBLAS).  The first product of a shape then takes
    up to ``max_ms_per_shape`` longer; worth it when shapes repeat (a fixed prefill portion, a steady
    decode batch), not for one-off shapes, so it is off unless asked for."""
    import torch.cuda.tunable as tunable
    tunable.enable(True)
    tunable.tuning_enable(True)
    tunable.set_max_tuning_duration(int(max_ms_per_shape))
    if not filename:
        import os
        from .library import _fallback_dir
        # this user's private folder under the temporary directory (refused if somebody else made it or may write it)
        filename = os.path.join(_fallback_dir(create=True), "tunableop.csv")
    tunable.set_filename(filename)     # choices are kept there and reused by later runs


def pause_library_gemm_tuning(paused: bool) -> None:
    """While paused, shapes already timed keep their chosen kernel and new shapes take the default."""
    import torch.cuda.tunable as tunable
    if tunable.is_enabled():
        tunable.tuning_enable(not paused)


def tile_weights(weight: torch.Tensor, order: Optional[torch.Tensor] = None, tile_rows: int = 16) -> torch.Tensor:
    """The tiled form of a bfloat16 ``weight`` [N, K] that the weight-streaming product reads in
    contiguous runs: a flat tensor of ceil(N / tile_rows) row tiles of ``tile_rows`` rows (even, 8 to 16) by
    cols64(K) k-values (zeros in the padding).  ``order`` (int32, a permutation of the row tiles, tiles of 16
    only): tile t of the copy is row tile order[t] of the weight."""
    _check(weight, "weight", (None, None), torch.bfloat16)
    N, K = weight.shape
    if K % 8:
        raise KernelError(f"tile_weights: K={K} must be a multiple of 8")
    if tile_rows not in TILE_ROWS or (order is not None and tile_rows != 16):
        raise KernelError(f"tile_weights: {tile_rows} rows to a tile (one of {TILE_ROWS}; 16 with a tile order)")
    mod = load_module("gemm_bf16")
    n_tiles = -(-N // tile_rows)
    if order is not None:
        _check(order, "order", (n_tiles,), torch.int32)
        if sorted(order.tolist()) != list(range(n_tiles)):
            raise KernelError("tile_weights: order is not a permutation of the weight's row tiles")
    out = empty((_tiled_size(N, K, tile_rows),), torch.bfloat16, weight)
    _call(mod, "ifx_tile_weights", (P, P, I, I, P, I, P), weight, out, N, K, order, tile_rows, _stream())
    return out


TILE_ROWS = (8, 10, 12, 14, 16)      # rows a tile of the copy may hold


def _tiled_size(N: int, K: int, tile_rows: int) -> int:
    return -(-N // tile_rows) * tile_rows * (-(-K // 64) * 64)


def choose_tile_rows(N: int) -> int:
    """Rows to a tile of a weight's streamed copy.  A workgroup of the products for few rows of x owns whole row
    tiles, and a compute unit can have only so many bytes on their way: a weight of 3,584 rows in tiles of 16
    gives 224 of the 256 units a tile and takes as long as one of 4,096 rows.  Where 16-row tiles leave units
    without one, the tiles are made as low as still gives every unit at most one (3,584 rows: 14; 2,048: 8).
    Measured at 1-64 rows of x: 3,584 x 18,944 takes 24.8 us instead of 25.9 at 8 rows, 2,048 x 11,008 16.3
    instead of 20.1 at 16 rows; weights with more tiles than units gain nothing from lower tiles or lose."""
    if N > 16 * COMPUTE_UNITS:
        return 16
    rows = -(-N // COMPUTE_UNITS)
    return min(16, max(8, rows + rows % 2))


class LinearWeight:
    """A projection's weight as the products want it: ``rows`` [N, K] as the model file has it, and for
    bfloat16 weights ``tiled``, the copy that products with few rows of x (decoding) stream from.  The
    copy doubles the weight's memory (see ``prepare_stacked`` for weights that are also rows of a larger one); it is left out when
    ``decode_weight_copy`` is off or when the card has no room for it, and products with few rows then read ``rows``."""

    __slots__ = ("rows", "tiled", "order", "tile_rows")

    def __init__(self, rows: torch.Tensor, tiled: Optional[torch.Tensor] = None, order: Optional[torch.Tensor] = None,
                 tile_rows: int = 16):
        # order: the copy's row-tile order, tile_rows: the rows to a tile of the copy (see tile_weights)
        self.rows, self.tiled, self.order, self.tile_rows = rows, tiled, order, tile_rows

    @property
    def shape(self):
        return self.rows.shape

    @property
    def dtype(self):
        return self.rows.dtype

    def part(self, start: int, stop: int) -> "LinearWeight":
        """Rows ``start`` .. ``stop`` - 1 as a weight of their own, sharing this one's memory (the copy too, where whole
        tiles of it hold just these rows)."""
        N, K = self.rows.shape
        tiled, tr = None, self.tile_rows
        if self.tiled is not None and self.order is None and start % tr == 0 and (stop % tr == 0 or stop == N):
            per_tile = tr * (-(-K // 64) * 64)
            tiled = self.tiled[start // tr * per_tile:-(-stop // tr) * per_tile]
        return LinearWeight(self.rows[start:stop], tiled, None, tr if tiled is not None else 16)


# Whether prepare_linear makes tiled copies, and how much memory it leaves free when it does.
decode_weight_copy = True
DECODE_COPY_RESERVE_BYTES = 8 << 30


def prepare_linear(weight: torch.Tensor, order: Optional[torch.Tensor] = None, tile_rows: int = 0) -> LinearWeight:
    """Wrap a projection's weight for ``linear`` / ``linear_swiglu``, with the tiled copy if wanted and possible
    (its row tiles in ``order``, if given, and then of 16 rows; else of ``tile_rows`` rows, 0: ``choose_tile_rows``)."""
    tiled = None
    if order is not None:
        tile_rows = 16
    elif tile_rows == 0:
        tile_rows = choose_tile_rows(weight.shape[0]) if weight.dim() == 2 else 16
    if (decode_weight_copy and weight.is_cuda and weight.dtype == torch.bfloat16 and weight.dim() == 2
            and weight.shape[1] % 8 == 0):
        free, _ = torch.cuda.mem_get_info(weight.device)
        if free >= weight.numel() * 2 + DECODE_COPY_RESERVE_BYTES:
            tiled = tile_weights(weight.contiguous(), order, tile_rows)
        else:
            log.warn("kernels", f"no room for the decode copy of a {tuple(weight.shape)} weight "
                                f"({free / 2**30:.1f} GiB free): decoding reads the plain rows")
    return LinearWeight(weight, tiled, order if tiled is not None else None, tile_rows if tiled is not None else 16)


def prepare_stacked(weights) -> Tuple[Optional[LinearWeight], list]:
    """(``weights`` [N_i, K] one below the other as one weight, each of them as a weight of its own), over the same rows.

    A part that would by itself have tiles as high as the whole's, and whose rows whole tiles of it hold, shares the whole's tiled copy (up to 2,048 rows in
    all, as a rule, every part).  The others have copies of their own, and the whole's is then one more, which it gets while a quarter of the card is free:
    copies of other weights may still have to be made.  The whole is None where it has no copy and a part has one."""
    rows = torch.cat(list(weights))
    ends = list(itertools.accumulate(w.shape[0] for w in weights))
    spans, height = list(zip([0] + ends, ends)), choose_tile_rows(rows.shape[0])
    shared = [choose_tile_rows(b - a) == height and a % height == 0 and (b % height == 0 or b == ends[-1]) for a, b in spans]
    free, total = torch.cuda.mem_get_info(rows.device)
    whole = prepare_linear(rows) if all(shared) or free >= total // 4 else LinearWeight(rows)
    parts = [whole.part(a, b) if s and whole.tiled is not None else prepare_linear(rows[a:b]) for s, (a, b) in zip(shared, spans)]
    return (None if whole.tiled is None and any(p.tiled is not None for p in parts) else whole), parts


class ScaledRows:
    """Rows of a normalised activation up to one factor per row: row t stands for
    ``rows[t] * rsqrt(sum(pieces[:, t]) / width + eps)``.  ``rows`` is bfloat16 [T <= 16, width] (the stream times
    the norm's weight), ``pieces`` float32 [n, 16] (sums of squares of the stream over runs of columns, one run
    per row tile of the product that made them; rows past T hold zeros).  A weight-streaming product that takes these multiplies its sums by the factor, which
    saves the norm a kernel of its own; ``linear_into_stream`` makes them."""

    __slots__ = ("rows", "pieces", "width", "eps", "norm_weight")

    def __init__(self, rows: torch.Tensor, pieces: torch.Tensor, width: int, eps: float,
                 norm_weight: Optional[torch.Tensor] = None):
        self.rows, self.pieces, self.width, self.eps = rows, pieces, int(width), float(eps)
        self.norm_weight = norm_weight      # the weight the rows were multiplied by: whose norm they stand for

    @property
    def shape(self):
        return self.rows.shape

    @property
    def dtype(self):
        return self.rows.dtype


class ScaledDelta:
    """A sub-block's output that is added to the stream times ``scale`` (a model's factor on every sub-block's output):
    ``value`` is a tensor or ``SliceSums``.  ``add_rmsnorm`` takes it as its delta; ``tensor()`` forms it for everyone
    else."""

    __slots__ = ("value", "scale")

    def __init__(self, value, scale: float):
        self.value, self.scale = value, float(scale)

    @property
    def shape(self):
        return self.value.shape

    def tensor(self) -> torch.Tensor:
        v = self.value.sum(torch.float32) if isinstance(self.value, SliceSums) else self.value.float()
        return v * self.scale


class DeltaSum:
    """Several things to be added to the stream, each times a factor: ``terms`` is a list of (value, factor), a value being a
    tensor [T, H], ``SliceSums`` or one vector [H] for all rows.  ``add_rmsnorm`` takes it as its delta and ``join_stream``
    as what is pending; nested sums and ``ScaledDelta`` are taken apart."""

    __slots__ = ("terms",)

    def __init__(self, terms):
        flat = []
        for v, s in terms:
            if isinstance(v, DeltaSum):
                flat += [(w, s * t) for w, t in v.terms]
            elif isinstance(v, ScaledDelta):
                flat.append((v.value, s * v.scale))
            else:
                flat.append((v, float(s)))
        self.terms = flat

    @classmethod
    def of(cls, *values) -> "DeltaSum":
        """The sum of ``values`` (None: nothing), each with factor 1."""
        return cls([(v, 1.0) for v in values if v is not None])

    def in_pieces(self, most: int) -> "DeltaSum":
        """The same terms in at most ``most`` tensors, vectors and single slices: where there are more, the ``SliceSums`` of the most slices
        are added up in float (products of narrow, deep weights have up to one for each pair of steps; experts one for each choice)."""
        terms, count = list(self.terms), lambda v: v.parts.shape[0] if isinstance(v, SliceSums) else 1
        while sum(count(v) for v, _ in terms) > most and any(count(v) > 1 for v, _ in terms):
            i = max(range(len(terms)), key=lambda k: count(terms[k][0]))
            terms[i] = (terms[i][0].sum(torch.float32), terms[i][1])
        return DeltaSum(terms)

    def tensor(self, like: torch.Tensor) -> torch.Tensor:
        """The sum as a float32 tensor of ``like``'s shape (for readers that add one tensor)."""
        out = torch.zeros_like(like, dtype=torch.float32)
        for v, s in self.terms:
            out += (v.sum(torch.float32) if isinstance(v, SliceSums) else v.float()) * s
        return out


class SplitRows:
    """Attention of a step of single rows [T, n_heads * width] (bfloat16) whose splits of the keys its reader joins: ``part_o`` float32
    [T, n_heads, splits, width] and ``part_ml`` [T, n_heads, splits, 2] as ``attention_rows`` leaves them, ``sinks`` float32 [n_heads] (or None) a
    score per head that joins the softmax's denominator.  ``headwise`` and ``diff_combine`` take it, which saves the launch that would join them."""

    __slots__ = ("part_o", "part_ml", "sinks")
    dtype = torch.bfloat16

    def __init__(self, part_o: torch.Tensor, part_ml: torch.Tensor, sinks: Optional[torch.Tensor] = None):
        self.part_o, self.part_ml, self.sinks = part_o, part_ml, sinks

    n_heads = property(lambda self: self.part_o.shape[1])
    n_splits = property(lambda self: self.part_o.shape[2])
    width = property(lambda self: self.part_o.shape[3])

    @property
    def shape(self):
        return torch.Size((self.part_o.shape[0], self.part_o.shape[1] * self.part_o.shape[3]))


SPLITS_READ_MAX = 32        # splits of a row that the readers of SplitRows take


class SliceSums:
    """A product left as partial sums over slices of K: it stands for ``parts.sum(0)`` (float32 [S, M, N], added in
    slice order).  ``add_rmsnorm`` takes it as its delta and ``rope_append`` as its q/k/v, which saves the kernel
    that would add the slices; ``sum()`` adds them for everyone else."""

    __slots__ = ("parts", "dtype")

    def __init__(self, parts: torch.Tensor, dtype: torch.dtype):
        self.parts, self.dtype = parts, dtype      # dtype: what the sum would be rounded to

    @property
    def shape(self):
        return self.parts.shape[1:]

    def sum(self, dtype: Optional[torch.dtype] = None) -> torch.Tensor:
        S, M, N = self.parts.shape
        out = torch.empty((M, N), dtype=dtype or self.dtype, device=self.parts.device)
        _call(load_module("gemm_wide"), "ifx_sum_slices", (P, P, I, I, LL, P),
              self.parts, out, _DT[out.dtype], S, M * N, _stream())
        return out


def _scale_args(x, columns: bool = False):
    """(rows, the four row-factor arguments of the kernels) of a tensor or a ``ScaledRows``; ``columns``: whose rows may be columns of wider ones."""
    if isinstance(x, ScaledRows):
        _check(x.pieces, "pieces", (None, 16), torch.float32)
        if not 1 <= x.pieces.shape[0] <= x.width:
            raise KernelError(f"scaled rows: {x.pieces.shape[0]} pieces for a width of {x.width}")
        if not (columns and columns_on_16_bytes(x.rows) and x.rows.shape[1] == x.width):
            _check(x.rows, "rows", (None, x.width), torch.bfloat16)
        if x.rows.shape[0] > 16:
            raise KernelError(f"scaled rows: {x.rows.shape[0]} rows, at most 16")
        return x.rows, (x.pieces.data_ptr(), x.pieces.shape[0], float(x.width), x.eps)
    return x, (0, 0, 0.0, 0.0)


def takes_scaled_rows(n_rows: int, weight) -> bool:
    """Whether ``linear`` / ``linear_swiglu`` / ``qkv_rope_append`` take ``ScaledRows`` of ``n_rows`` rows with this weight."""
    if not isinstance(weight, LinearWeight):
        return False
    N, K = weight.rows.shape
    return (weight.rows.dtype == torch.bfloat16 and n_rows <= 16
            and _small_m_kernel(n_rows, N, K, weight.tiled is not None) in ("skinny", "wide"))


def adds_into_stream(n_rows: int, weight, norm_weight: torch.Tensor, single_tokens: bool = True) -> bool:
    """Whether a product of this shape is best added to the stream by ``linear_into_stream``, which takes it then.

    Where 9 to 16 rows times a deep weight of up to 2,048 rows go to the ring in slices of K, they and the norm that adds the slices are faster (us of down and the
    product behind it, into the stream : slices and norm, at 9, 12 and 16 rows: 896 x 4,864 12.0, 13.1, 14.1 : 11.1,
    11.6, 11.8, 1,024 x 4,224 12.1, 13.1, 13.9 : 11.4, 11.5, 11.8, 1,536 x 8,960 17.3, 18.1, 19.3 : 15.6, 16.0, 16.0, 2,048 x 11,008 33.5, 34.8, 34.4 : 30.6, 30.9, 30.4;
    but 2,560 x 9,728 22.3, 21.0, 23.5 : 22.8, 21.8, 22.4, 3,584 x 18,944 38.4, 41.8, 47.4 : 40.6, 41.3, 42.0, and at 8 rows all but one slower).  So in steps of single tokens, which
    graphs replay (ms for 48 tokens of 16 requests at the 0.5B, 1.5B and 3B shapes 42.0, 68.9, 102.7 : 39.7, 65.3, 97.6); a prompt's step is run launch by launch and waits for the
    host, to whom the norm and the sums are a launch and an allocation more a layer (12 tokens 1.48, 1.72, 2.20 : 1.70, 2.00, 2.53)."""
    if not _into_stream_takes(n_rows, weight, norm_weight):
        return False
    if n_rows < RING_FEW_MIN_ROWS or weight.tiled is None or not single_tokens:
        return True
    N, K = weight.rows.shape
    return N > RING_FEW_STREAM_MAX_N or not _few_in_slices(n_rows, N, K, weight.tile_rows)


def _into_stream_takes(n_rows: int, weight, norm_weight: torch.Tensor) -> bool:
    # (without a norm's weight: a reader that takes partial sums but keeps the addition to itself)
    if n_rows > 16 or norm_weight is None or not isinstance(weight, LinearWeight) or weight.order is not None:
        return False
    rows = weight.rows
    N, K = rows.shape
    return N % 4 == 0 and rows.dtype == torch.bfloat16 and _small_m_kernel(n_rows, N, K, weight.tiled is not None) == "skinny"


def linear_into_stream(x: torch.Tensor, weight: LinearWeight, stream: torch.Tensor, norm_weight: torch.Tensor,
                       eps: float, mult: float = 1.0) -> ScaledRows:
    """``stream`` [M <= 16, N] (float32) += ``mult`` * x [M, K] W^T in place, as the product's epilogue, which also prepares
    the RMS norm that follows (weight ``norm_weight`` [N]): returns its rows up to the factor per row."""
    _check(x, "x", (None, None), torch.bfloat16)
    M, K = x.shape
    N = weight.rows.shape[0]
    if not _into_stream_takes(M, weight, norm_weight) or weight.rows.shape[1] != K:
        raise KernelError(f"linear_into_stream: not for {M} rows times a {tuple(weight.rows.shape)} weight")
    _check(stream, "stream", (M, N), torch.float32)
    _check(norm_weight, "norm_weight", (N,))
    rows = empty((M, N), torch.bfloat16, x)
    tile_rows = 16 if weight.tiled is None else weight.tile_rows
    pieces = empty((-(-N // tile_rows), 16), torch.float32, x)    # one piece per row tile
    w = weight.rows if weight.tiled is None else weight.tiled
    _call(load_module("gemm_bf16"), "ifx_skinny_gemm", _SKINNY_ARGS,
          x, w, 0, DT_F32, M, N, K, 0, 0, 0, 2, 0 if weight.tiled is None else tile_rows, 0,
          0, 0, 0.0, 0.0, stream, norm_weight, 1 if norm_weight.dtype == torch.float32 else 0, rows,
          pieces, float(mult), 0, 0, _stream())
    return ScaledRows(rows, pieces, N, eps, norm_weight)


_SKINNY_ARGS = (P, P, P, I, I, I, I, I, I, I, I, I, P, P, I, F, F, P, P, I, P, P, F, I, I, P)


def pair_tile_order(n_heads: int, head_dim: int) -> list:
    """Row-tile order of a projection whose rows are ``n_heads`` heads of ``head_dim`` (a multiple of 32) that
    puts the two halves of 16 split-half rotation pairs into consecutive tiles: for head h and j < d / 32,
    tiles h d/16 + j and h d/16 + j + d/32.  What ``qkv_rope_append`` expects of its tiled copy."""
    per, half = head_dim // 16, head_dim // 32
    return [h * per + j + s * half for h in range(n_heads) for j in range(half) for s in (0, 1)]


def qkv_rope_append(x: torch.Tensor, weight: LinearWeight, bias: Optional[torch.Tensor], slots: Optional[torch.Tensor],
                    cos: torch.Tensor, sin: torch.Tensor, n_heads: int, n_kv_heads: int, head_dim: int,
                    k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor], page_size: int,
                    waves: int = 0, unroll: int = 0) -> torch.Tensor:
    """For up to 16 tokens: q, k, v = x W^T + bias from the pair-ordered tiled copy of the concatenated
    weight, q and k rotated (split-half pairs over the whole head, table cos/sin [M, d/2]), k and v written
    into the paged cache at ``slots``, q returned [M, nH, d] -- one kernel, the rotation and the cache
    write being the product's epilogue.  With ``slots`` None the weight holds the query rows only.
    ``x`` may be ``ScaledRows``."""
    x, scale = _scale_args(x)
    _check(x, "x", (None, None), torch.bfloat16)
    M, K = x.shape
    heads = n_heads + (2 * n_kv_heads if slots is not None else 0)
    if weight.tiled is None or weight.order is None or tuple(weight.rows.shape) != (heads * head_dim, K):
        raise KernelError(f"qkv_rope_append: needs the pair-ordered tiled copy of a [{heads * head_dim}, {K}] weight")
    if M > 16 or head_dim % 32 or K % 8:
        raise KernelError(f"qkv_rope_append: M={M} must be <= 16, head_dim={head_dim} a multiple of 32, K={K} of 8")
    _check(cos, "cos", (M, head_dim // 2), torch.float32)
    _check(sin, "sin", (M, head_dim // 2), torch.float32)
    if bias is not None:
        _check(bias, "bias", (heads * head_dim,))
        if bias.data_ptr() % 16:          # (a part of a larger tensor: the kernel reads four elements at a time)
            bias = bias.clone()
    if slots is not None:
        _check(slots, "slots", (M,), torch.int32)
        _check(k_cache, "k_cache", (None, n_kv_heads, page_size, head_dim), torch.bfloat16)
        _check(v_cache, "v_cache", (k_cache.shape[0], n_kv_heads, head_dim, page_size), torch.bfloat16)
    q = empty((M, n_heads, head_dim), torch.bfloat16, x)
    _call(load_module("gemm_bf16"), "ifx_qkv_rope", (P, P, I, I, P, I, P, P, P, I, I, I, I, P, P, P, I, I, P, I, F, F, P),
          x, weight.tiled, M, K, bias, _dt(bias) if bias is not None else 0, slots,
          cos, sin, n_heads, n_kv_heads, head_dim, page_size, q, k_cache,
          v_cache, waves, unroll, *scale, _stream())
    return q


@functools.lru_cache(maxsize=4096)
def _narrow_f32(M: int, N: int) -> bool:
    return load_module("gemm_f32").fn("ifx_gemm_f32_narrow_slices", (I, I))(M, N) > 0


def qkv_rope_f32_takes(x: torch.Tensor, weight, bias: Optional[torch.Tensor]) -> bool:
    """Whether ``qkv_rope_f32`` takes these rows, weight and bias: where ``gemm_f32`` has its kernel for up to 8 rows."""
    if x.dtype != torch.float32 or not 0 < x.shape[0] <= 8 or not isinstance(weight, LinearWeight) or weight.rows.dtype != torch.float32:
        return False
    N, K = weight.rows.shape
    return (K % 4 == 0 and _narrow_f32(x.shape[0], N) and (bias is None or bias.dtype == torch.float32) and x.is_contiguous() and x.data_ptr() % 16 == 0
            and weight.rows.data_ptr() % 16 == 0)


def qkv_rope_f32(x: torch.Tensor, weight: LinearWeight, bias: Optional[torch.Tensor], slots: Optional[torch.Tensor], cos: torch.Tensor, sin: torch.Tensor,
                 n_heads: int, n_kv_heads: int, head_dim: int, k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor], page_size: int) -> torch.Tensor:
    """``qkv_rope_append`` in 32 bits, for up to 8 rows: the bits of ``linear`` and ``rope_append`` (split-half pairs over the whole head, values as wide as
    keys)."""
    if not qkv_rope_f32_takes(x, weight, bias):
        raise KernelError(f"qkv_rope_f32: not for {x.shape[0]} rows times a {tuple(weight.rows.shape)} weight")
    (M, K), N = x.shape, weight.rows.shape[0]
    n_kv = n_kv_heads if slots is not None else 0
    if weight.rows.shape[1] != K or head_dim % 2 or N != (n_heads + 2 * n_kv) * head_dim:
        raise KernelError(f"qkv_rope_f32: a {tuple(weight.rows.shape)} weight for rows of {K} and {n_heads} + {n_kv} heads of {head_dim}")
    _check(cos, "cos", (M, head_dim // 2), torch.float32)
    _check(sin, "sin", (M, head_dim // 2), torch.float32)
    if bias is not None:
        _check(bias, "bias", (N,), torch.float32)
    if slots is not None:
        _check(slots, "slots", (M,), torch.int32)
        _check(k_cache, "k_cache", (None, n_kv, page_size, head_dim), torch.float32)
        _check(v_cache, "v_cache", (k_cache.shape[0], n_kv, head_dim, page_size), torch.float32)
    else:
        k_cache = v_cache = None
    q = empty((M, n_heads, head_dim), torch.float32, x)
    _call(load_module("gemm_f32"), "ifx_qkv_rope_f32", (P, P, P, P, I, I, I, P, P, P, I, I, I, I, P, P, P),
          x, weight.rows, bias, q, M, N, K, slots, cos, sin, n_heads, n_kv, head_dim, page_size, k_cache, v_cache, _stream())
    return q


def columns_on_16_bytes(x) -> bool:
    """Whether ``x`` is a bfloat16 matrix on the GPU whose rows are columns of wider rows, each run of eight on 16 bytes: what
    ``skinny_gemm`` reads where it lies."""
    # (asked on every launch: whole rows leave at once)
    return (type(x) is torch.Tensor and not x.is_contiguous() and x.is_cuda and x.dtype == torch.bfloat16 and x.dim() == 2
            and x.stride(1) == 1 and x.stride(0) >= x.shape[1] and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0)


def skinny_gemm(x: torch.Tensor, weight: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16,
                nt: int = 0, waves: int = 0, unroll: int = 0, swiglu_pairs: bool = False,
                tiled: Optional[torch.Tensor] = None, order: Optional[torch.Tensor] = None, tile_rows: int = 16,
                act: int = ACT_SILU, plain_act: Optional[int] = None) -> torch.Tensor:
    """bfloat16 x [M <= 64, K] times bfloat16 ``weight`` [N, K] transposed on the matrix cores, float
    accumulation, output bfloat16 or float32.  ``nt``, ``waves``, ``unroll`` = 0 lets the kernel choose.
    With ``swiglu_pairs`` the weight's rows alternate gate and up and the output is act(gate) * up [M, N/2] (``act``:
    ACT_SILU or ACT_GELU_TANH).  With ``tiled`` (``tile_weights(weight, order, tile_rows)``) the kernel streams that copy instead of the rows.
    ``x`` may be ``ScaledRows``, or a tensor whose rows are further apart than K (columns of wider rows, on 16 bytes).
    ``plain_act`` (ACT_RELU_SQUARED, ACT_GELU_TANH; bfloat16 output): the activation of a feed-forward without a gate on the
    float sums."""
    x, scale = _scale_args(x, True)
    apart = 0
    if columns_on_16_bytes(x):
        apart = x.stride(0)
    else:
        _check(x, "x", (None, None), torch.bfloat16)
    M, K = x.shape
    _check(weight, "weight", (None, K), torch.bfloat16)
    N = weight.shape[0]
    if plain_act is not None and (plain_act not in _PLAIN_EPILOGUE or swiglu_pairs or order is not None or out_dtype != torch.bfloat16):
        raise KernelError(f"skinny_gemm: activation {plain_act} is no epilogue of this product")
    epilogue = _GATED_EPILOGUE[act] if swiglu_pairs else (_PLAIN_EPILOGUE[plain_act] if plain_act is not None else 0)
    if tiled is not None:
        if tile_rows not in TILE_ROWS or (order is not None and tile_rows != 16):
            raise KernelError(f"skinny_gemm: {tile_rows} rows to a tile (one of {TILE_ROWS}; 16 with a tile order)")
        _check(tiled, "tiled", (_tiled_size(N, K, tile_rows),), torch.bfloat16)
    if M > SKINNY_MAX_M or K % 8:
        raise KernelError(f"skinny_gemm: M={M} must be <= {SKINNY_MAX_M} and K={K} a multiple of 8")
    if swiglu_pairs and N % 2:
        raise KernelError("skinny_gemm: gate/up pairs need an even number of weight rows")
    out = empty((M, N // 2 if swiglu_pairs else N), out_dtype, x)
    if order is not None and (tiled is None or swiglu_pairs):
        raise KernelError("skinny_gemm: a tile order goes with a tiled copy and a plain product")
    _call(load_module("gemm_bf16"), "ifx_skinny_gemm", _SKINNY_ARGS,
          x, (weight if tiled is None else tiled), out, _DT[out_dtype], M, N, K, nt, waves,
          unroll, epilogue, 0 if tiled is None else tile_rows, order, *scale, 0, 0, 0, 0, 0,
          1.0, 0, apart, _stream())
    return out


def wide_gemm(x, weight: LinearWeight, out_dtype: torch.dtype = torch.bfloat16, waves: int = 0,
              slices: int = 0, swiglu_pairs: bool = False, keep_slices: bool = False, act: int = ACT_SILU):
    """bfloat16 x [M <= 128, K] times ``weight`` transposed from its tiled copy, x shared through LDS by the waves
    of a workgroup: the product for 17-64 rows, for 65-128 rows of weights with few rows, and for 9-16 rows of large
    tall weights.  ``waves`` (4-16 per workgroup, 8 beyond 64 rows; one tile of weight rows each) and ``slices`` of K
    (added in a fixed order): 0 lets the kernel choose, and with both 0 the ring of slots is taken where it is faster (``ring_takes``).  With ``keep_slices`` a product of several slices comes back as
    ``SliceSums``.  ``x`` may be ``ScaledRows`` (up to 16 rows)."""
    x, scale = _scale_args(x)
    _check(x, "x", (None, None), torch.bfloat16)
    M, K = x.shape
    N = weight.rows.shape[0]
    # (more than 16 rows carry no factor)
    ring = waves == 0 and slices == 0 and weight.tiled is not None and K % 8 == 0 and x.data_ptr() % 16 == 0
    if ring and not swiglu_pairs and _ring_in_one_slice(M, N, K, weight.tile_rows, keep_slices):
        return ring_gemm(x, weight, out_dtype, slices=1)
    if ring and ring_takes(M, N, K, weight.tile_rows, swiglu_pairs) and not (swiglu_pairs and (N % 2 or weight.order is not None)):
        return ring_gemm(x, weight, out_dtype, swiglu_pairs=swiglu_pairs, keep_slices=keep_slices, act=act)
    if weight.tiled is None or weight.rows.shape[1] != K or weight.rows.dtype != torch.bfloat16:
        raise KernelError(f"wide_gemm: needs the tiled copy of a bfloat16 [N, {K}] weight")
    if M > WIDE_MAX_M or K % 8:
        raise KernelError(f"wide_gemm: M={M} must be <= {WIDE_MAX_M} and K={K} a multiple of 8")
    if swiglu_pairs and (N % 2 or weight.order is not None):
        raise KernelError("wide_gemm: gate/up pairs need an even number of weight rows in their natural order")
    mod = load_module("gemm_wide")
    if _tiled_size(N, K, weight.tile_rows) != weight.tiled.numel():
        raise KernelError(f"wide_gemm: the copy is not that of a [{N}, {K}] weight in tiles of {weight.tile_rows} rows")
    plan = _wide_plan(M, N, K, waves, slices, 1 if swiglu_pairs else 0, weight.tile_rows)
    n_waves, n_slices = plan // 256, plan % 256
    part = empty((n_slices, M, N), torch.float32, x) if n_slices > 1 else None
    keep = keep_slices and n_slices > 1
    out = None if keep else empty((M, N // 2 if swiglu_pairs else N), out_dtype, x)
    _call(mod, "ifx_wide_gemm", (P, P, P, I, P, I, I, I, I, I, I, P, I, P, I, F, F, I, I, P),
          x, weight.tiled, out, _DT[out_dtype], part, M, N, K, n_waves, n_slices,
          _GATED_EPILOGUE[act] if swiglu_pairs else 0, weight.order, weight.tile_rows, *scale, 0, 0, _stream())
    return SliceSums(part, out_dtype) if keep else out


@functools.lru_cache(maxsize=4096)
def _wide_plan(M: int, N: int, K: int, waves: int, slices: int, pairs: int, tile_rows: int) -> int:
    """waves * 256 + slices of the product that shares x through LDS."""
    return load_module("gemm_wide").fn("ifx_wide_gemm_plan", (I, I, I, I, I, I, I))(M, N, K, waves, slices, pairs, tile_rows)


def ring_gemm(x: torch.Tensor, weight: LinearWeight, out_dtype: torch.dtype = torch.bfloat16, row_tiles: int = 0, slices: int = 0,
              swiglu_pairs: bool = False, keep_slices: bool = False, act: int = ACT_SILU, plain_act: Optional[int] = None):
    """bfloat16 x [M <= 64, K] times ``weight`` transposed from its tiled copy, both through a ring of slots in LDS.  ``row_tiles`` (1 to 8)
    of the weight to a workgroup and ``slices`` of K: 0 chooses (``ring_plan``); ``keep_slices`` and the gated epilogue as for
    ``wide_gemm``, ``plain_act`` (up to 16 rows) as for ``skinny_gemm``."""
    if plain_act is not None and (plain_act not in _PLAIN_EPILOGUE or swiglu_pairs or weight.order is not None or out_dtype != torch.bfloat16 or x.shape[0] > 16):
        raise KernelError(f"ring_gemm: activation {plain_act} is no epilogue of this product")
    _check(x, "x", (None, None), torch.bfloat16)
    M, K = x.shape
    N = weight.rows.shape[0]
    if weight.tiled is None or weight.rows.shape[1] != K or weight.rows.dtype != torch.bfloat16 or K % 8:
        raise KernelError(f"ring_gemm: needs the tiled copy of a bfloat16 [N, {K}] weight")
    if swiglu_pairs and (N % 2 or weight.order is not None):
        raise KernelError("ring_gemm: gate/up pairs need an even number of weight rows in their natural order")
    if _tiled_size(N, K, weight.tile_rows) != weight.tiled.numel():
        raise KernelError(f"ring_gemm: the copy is not that of a [{N}, {K}] weight in tiles of {weight.tile_rows} rows")
    row_tiles, steps = ring_plan(M, N, K, weight.tile_rows, swiglu_pairs or plain_act is not None or slices == 1, row_tiles, slices)
    n_slices = -(-(-(-K // 128)) // steps)
    part = empty((n_slices, M, N), torch.float32, x) if n_slices > 1 else None
    out = None if n_slices > 1 else empty((M, N // 2 if swiglu_pairs else N), out_dtype, x)
    _call(load_module("gemm_ring"), "ifx_ring_gemm", (P, P, P, I, P, I, I, I, I, I, I, I, P, I, P),
          x, weight.tiled, out, _DT[out_dtype], part, M, N, K, row_tiles, n_slices, steps,
          _GATED_EPILOGUE[act] if swiglu_pairs else (_PLAIN_EPILOGUE[plain_act] if plain_act is not None else 0), weight.order,
          weight.tile_rows, _stream())
    if n_slices == 1:
        return out
    sums = SliceSums(part, out_dtype)
    return sums if keep_slices else sums.sum()


RING_DEEP_STEPS = 48          # steps of 128 k-values from which a slice's own traffic, not its start, sets the row tiles to a workgroup


@functools.lru_cache(maxsize=4096)
def ring_plan(M: int, N: int, K: int, tile_rows: int, one_slice: bool, row_tiles: int = 0, slices: int = 0) -> Tuple[int, int]:
    """(row tiles to a workgroup, steps of 128 k-values to a slice): about one workgroup to each of the 256 compute units.

    Weights that are cut into slices of K: of up to 128 tiles of 16 rows (or pairs of 8, which the kernel joins: up to 2,048 rows) K is cut into four, or more where that leaves compute
    units without a workgroup; a workgroup takes one tile, two where K is deep or there are 96 tiles and 17 rows (us by one, two and four tiles: 1,024 x 4,224 at 16 rows 4.3, 4.9,
    6.3, 2,048 x 4,096 at 32 6.8, 6.3, 6.8, 1,536 x 8,960 at 16 9.0, 7.5, 8.4, at 64 13.0, 10.3, and 10.1 with twice the partial sums to read).  Of more tiles a workgroup
    takes two where K is short (us by one, two, four and eight: 2,560 x 2,048 at 17 rows 6.3, 5.2, 5.7, 6.8, at 64 8.5, 7.1, 7.4, 7.8) and, where it is deep,
    four up to 32 rows and eight beyond, whose x is read half as often (3,584 x 18,944 at 17 rows 40.4, 25.2, 25.8, 26.8, at 64 52.9, 39.4, 32.6, 29.5)."""
    steps = -(-K // 128)
    if not one_slice and row_tiles <= 0 and slices <= 0 and -(-N // (16 if tile_rows == 8 else tile_rows)) <= 128:
        n_tiles, deep = -(-N // (16 if tile_rows == 8 else tile_rows)), steps >= RING_DEEP_STEPS
        row_tiles = 2 if deep or (M > 16 and n_tiles >= 96) else 1
        slices = max(1, min(max(4, COMPUTE_UNITS // -(-n_tiles // row_tiles)), steps // 2))
        per = -(-steps // slices)
        return (2 * row_tiles if tile_rows == 8 and per < steps else row_tiles), per
    n_tiles = -(-N // tile_rows)
    if row_tiles <= 0:
        row_tiles = -(-n_tiles // COMPUTE_UNITS) if one_slice else 2 if steps < RING_DEEP_STEPS else 4 if M <= 32 else 8
        row_tiles = min(8, row_tiles)
    if one_slice:
        slices = 1
    elif slices <= 0:
        slices = max(1, min(COMPUTE_UNITS // -(-n_tiles // row_tiles), steps // 2))
    return row_tiles, -(-steps // min(slices, steps))


@functools.lru_cache(maxsize=4096)
def ring_takes(M: int, N: int, K: int, tile_rows: int, one_slice: bool) -> bool:
    """Whether 17 to 64 rows go to ``ring_gemm`` instead of ``wide_gemm``: where a row of workgroups holds the weight's row tiles, up to
    six to a workgroup for gate/up and one a compute unit for weights that are cut into slices (us at 17 / 32 / 64 rows, wide : ring)
        gate/up 9,728 x 896 9.4 : 6.8, 9.7 : 7.2, 10.7 : 8.6      17,920 x 1,536 14.4 : 13.4, 14.9 : 13.4, 16.9 : 14.7
                22,016 x 2,048 22.2 : 19.1, 22.2 : 19.3, 22.1 : 20.0, but 37,888 x 3,584 45.1 : 46.8, 44.1 : 47.5, 50.8 : 54.2
        896 x 4,864 6.6 : 5.0, 6.7 : 5.0, 9.0 : 6.5     1,536 x 8,960 10.5 : 7.3, 10.3 : 8.0, 13.6 : 10.3    1,024 x 1,024 4.3 : 3.1, 4.5 : 3.2, 5.6 : 3.8
        3,584 x 18,944 25.5 : 24.1, 25.6 : 24.5, 31.0 : 28.3     2,560 x 2,048 5.3 : 5.2, 5.8 : 5.6, 7.6 : 7.1, but 4,608 x 3,584 8.5 : 8.8, 9.1 : 9.2, 11.2 : 11.1."""
    return 17 <= M <= SKINNY_MAX_M and -(-N // tile_rows) <= (6 if one_slice else 1) * COMPUTE_UNITS and K < 1 << 20


@functools.lru_cache(maxsize=4096)
def _ring_in_one_slice(M: int, N: int, K: int, tile_rows: int, keep_slices: bool) -> bool:
    """Whether ``wide_gemm`` hands 17 to 64 rows times a weight that it would cut into slices of K to ``ring_gemm`` uncut: up to 4,096 k-values
    where nobody adds slices on the way, up to 2,048 where the reader does (us at 17 / 32 / 64 rows: slices and their sum, slices alone, uncut)
        6,208 x 2,048 10.9, 8.2, 7.3 / 11.9, 8.5, 7.9 / 15.2, 10.6, 10.6     12,288 x 2,048 16.7, 14.3, 10.8 / 17.1, 14.4, 11.1 / 21.2, 17.1, 13.5
        4,608 x 3,584 12.4, 8.7, 9.9 / 13.3, 9.2, 11.2 / 17.2, 11.3, 15.3     3,104 x 1,024 6.7, 4.7, 4.7 / 6.9, 4.9, 5.0 / 8.4, 6.2, 6.4
        4,352 x 2,048 10.5, 7.4, 7.0 / 11.6, 7.9, 7.6 / 14.7, 9.9, 10.3     4,096 x 4,096 10.8, 8.2, 9.6 / 10.9, 8.8, 9.9 / 13.7, 11.3, 13.9."""
    tiles = -(-N // tile_rows)
    if not 17 <= M <= SKINNY_MAX_M or K % 8 or N <= 2048 or tiles > 6 * COMPUTE_UNITS:
        return False
    return tiles > COMPUTE_UNITS and K <= 2048 if keep_slices else K <= 4096


RING_FEW_MIN_ROWS = 9            # (up to 8 rows x is little to read beside W)
RING_FEW_MIN_SLICED_K = 4096
RING_FEW_STREAM_MAX_N = 2048         # (see ``adds_into_stream``)


def _few_in_slices(n_rows: int, N: int, K: int, tile_rows: int) -> bool:
    """Whether so many rows times a weight that would go to the product whose waves split K go to ``ring_gemm`` in slices of K instead, where their reader adds
    the slices (see ``ring_takes_few``; ``adds_into_stream`` asks for every product of a step, so this is a few comparisons)."""
    return RING_FEW_MIN_ROWS <= n_rows <= 16 and -(-N // tile_rows) <= COMPUTE_UNITS and RING_FEW_MIN_SLICED_K <= K < 1 << 20


def ring_takes_few(x, weight, keep_slices: bool = False) -> int:
    """Whether 9 to 16 rows that would go to the product whose waves each read x from the L2 go to ``ring_gemm``, whose workgroups read it
    once: 1 in one slice of K, 2 in slices whose sum the caller takes, 0 not (us at 9 and 16 rows, that product : this one)
        one slice, weights of 2,049 to 12,288 rows and up to 4,096 k-values: 8,448 x 2,048 10.0, 12.9 : 9.1, 9.4     6,272 x 2,048 8.2, 9.4 : 7.5, 7.7
            11,264 x 2,048 12.2, 12.4 : 11.1, 10.7     9,728 x 896 6.8, 7.1 : 6.6, 6.8     4,224 x 1,024 5.6, 5.9 : 5.5, 5.5     3,136 x 1,024 4.4, 4.8 :
            4.2, 4.3, but 17,920 x 1,536 11.9, 13.9 : 12.9, 12.6, 22,016 x 2,048 16.8, 17.5 : 18.1, 17.7, 2,048 x 8,448 12.9, 14.4 : 13.6, 13.4
        slices, a row tile for a compute unit at most and 4,096 k-values or more: 2,048 x 8,448 12.9, 14.4 : 9.0, 8.7     1,024 x 4,224 7.2, 8.6 : 4.2, 4.3
            2,048 x 5,632 9.7, 10.9 : 8.1, 8.2     1,536 x 8,960 12.3, 13.7 : 7.5, 7.6     3,584 x 18,944 26.2, 32.8 : 24.5, 24.2, but 2,048 x 2,048 5.4, 5.8 :
            4.5, 4.5 and a sum for the reader to form."""
    if x.shape[0] < RING_FEW_MIN_ROWS:              # (most steps that ask)
        return 0
    if not isinstance(weight, LinearWeight) or isinstance(x, ScaledRows) or weight.tiled is None or weight.rows.dtype != torch.bfloat16 \
            or x.dtype != torch.bfloat16 or not x.is_contiguous() or x.data_ptr() % 16:
        return 0
    (M, K), N = x.shape, weight.rows.shape[0]
    if not RING_FEW_MIN_ROWS <= M <= 16 or K % 8 or K != weight.rows.shape[1] or _small_m_kernel(M, N, K, True) != "skinny":
        return 0
    if keep_slices and _few_in_slices(M, N, K, weight.tile_rows):
        return 2
    tiles = -(-N // weight.tile_rows)
    return 1 if 2048 < N and tiles <= 3 * COMPUTE_UNITS and K <= RING_FEW_MIN_SLICED_K else 0


def leaves_few_rows_in_sums(x, weight) -> bool:
    """Whether ``linear`` with ``keep_slices`` leaves these up to 16 rows times ``weight`` as partial sums in float."""
    if x.shape[0] < 8:              # (neither of the two kernels that cut K takes fewer)
        return False
    N, K = weight.rows.shape
    return ring_takes_few(x, weight, True) == 2 or (weight.tiled is not None and N < WIDE_FEW_ROWS_MIN_N and _small_m_kernel(x.shape[0], N, K, True) == "wide")


def streams_weight(n_rows: int, weight) -> bool:
    """Whether ``linear`` of ``n_rows`` rows with this weight goes to the kernels that stream a weight for few rows (whose
    float sums cost nothing more than rounded ones) or, in 32-bit, to the 32-bit kernel, and not to the library."""
    rows = weight.rows if isinstance(weight, LinearWeight) else weight
    if rows.dtype == torch.float32:
        return True
    has_tiled = isinstance(weight, LinearWeight) and weight.tiled is not None
    return _small_m_kernel(n_rows, rows.shape[0], rows.shape[1], has_tiled) is not None


def _blocks_kernel(n_rows: int, weight, block_rows: int) -> Optional[str]:
    if not (isinstance(weight, LinearWeight) and weight.dtype == torch.bfloat16 and weight.tiled is not None and weight.order is None
            and weight.tile_rows == 16 and block_rows % 16 == 0 and weight.rows.shape[1] % 8 == 0):
        return None
    if n_rows <= 16:
        return "skinny"
    return "wide" if n_rows <= SKINNY_MAX_M and block_rows % 128 == 0 else None


def takes_blocks(n_rows: int, weight, block_rows: int) -> bool:
    """Whether ``linear_blocks`` takes this shape."""
    return _blocks_kernel(n_rows, weight, block_rows) is not None


def linear_blocks(x: torch.Tensor, weight: "LinearWeight", block_rows: int, out_dtype: torch.dtype = torch.bfloat16) -> torch.Tensor:
    """Several products of few rows in one launch: ``x`` [n, M, K] holds n inputs, ``weight`` [N, K] (with its copy in tiles of
    16 rows) n blocks of rows, all of ``block_rows`` except the last, which is what remains; block b's columns of the result
    [M, N] are x[b] times block b transposed."""
    _check(x, "x", (None, None, None), torch.bfloat16)
    n, M, K = x.shape
    kind = _blocks_kernel(M, weight, block_rows)
    N = weight.rows.shape[0]
    if kind is None or weight.rows.shape[1] != K or not (n - 1) * block_rows < N:
        raise KernelError(f"linear_blocks: not for {n} inputs of {M} rows times a {tuple(weight.rows.shape)} weight in blocks of {block_rows}")
    tiles = block_rows // 16
    if kind == "skinny":
        out = empty((M, N), out_dtype, x)
        _call(load_module("gemm_bf16"), "ifx_skinny_gemm", _SKINNY_ARGS, x, weight.tiled, out, _DT[out_dtype],
              M, N, K, 0 if tiles % 2 == 0 else 1, 0, 0, 0, 16, 0, 0, 0, 0.0, 0.0, 0, 0, 0, 0, 0, 1.0, tiles, n, _stream())
        return out
    mod = load_module("gemm_wide")
    plan = _wide_plan(M, N, K, 8, 0, 0, 16)
    n_slices = plan % 256
    part = empty((n_slices, M, N), torch.float32, x) if n_slices > 1 else None
    out = empty((M, N), out_dtype, x)
    _call(mod, "ifx_wide_gemm", (P, P, P, I, P, I, I, I, I, I, I, P, I, P, I, F, F, I, I, P),
          x, weight.tiled, out, _DT[out_dtype], part, M, N, K, 8, n_slices, 0, 0, 16, 0, 0, 0.0, 0.0,
          tiles, n, _stream())
    return out


def staged_gemm(x: torch.Tensor, weight: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16,
                slices: int = 0, unroll: int = 0, swiglu_pairs: bool = False, act: int = ACT_SILU) -> torch.Tensor:
    """The same product as skinny_gemm with x staged in LDS and shared by the waves of a workgroup
    (64 weight rows per workgroup, K cut into ``slices``; 0 lets the kernel choose)."""
    _check(x, "x", (None, None), torch.bfloat16)
    M, K = x.shape
    _check(weight, "weight", (None, K), torch.bfloat16)
    N = weight.shape[0]
    if M > SKINNY_MAX_M or K % 8:
        raise KernelError(f"staged_gemm: M={M} must be <= {SKINNY_MAX_M} and K={K} a multiple of 8")
    if swiglu_pairs and N % 2:
        raise KernelError("staged_gemm: gate/up pairs need an even number of weight rows")
    mod = load_module("gemm_bf16")
    n_slices = 1 if swiglu_pairs else mod.fn("ifx_staged_gemm_slices", (I, I, I, I))(M, N, K, slices)
    part = empty((n_slices, M, N), torch.float32, x) if n_slices > 1 else None
    out = empty((M, N // 2 if swiglu_pairs else N), out_dtype, x)
    _call(mod, "ifx_staged_gemm", (P, P, P, I, P, I, I, I, I, I, I, P),
          x, weight, out, _DT[out_dtype], part, M, N, K, slices, unroll,
          _GATED_EPILOGUE[act] if swiglu_pairs else 0, _stream())
    return out


def linear(x: torch.Tensor, weight, out_dtype: Optional[torch.dtype] = None, keep_slices: bool = False):
    """x [M, K] times ``weight`` [N, K] transposed (a tensor or a ``LinearWeight``), chosen by the weight's
    type and by M.  With ``keep_slices`` the result may be ``SliceSums`` (the caller hands it to ``add_rmsnorm`` or
    ``rope_append``, or calls its ``sum()``).  ``x`` is contiguous, or in bfloat16 columns of wider rows on 16 bytes
    (``columns_on_16_bytes``).

    A float32 weight takes the true 32-bit kernel whatever the activation's type.  A bfloat16
    weight with bfloat16 activations takes the weight-streaming kernel for up to 64 rows and the
    library product with float accumulation beyond, as the reference does for every dense
    projection (runtime/backends/cuda/native/cublas_gemm.cpp:99-117).  float32 output (logits)
    always comes from float accumulators, never through a bfloat16 rounding.
    """
    tiled = order = None
    tile_rows = 16
    if isinstance(x, ScaledRows) and not takes_scaled_rows(x.shape[0], weight):
        raise KernelError(f"linear: scaled rows are not taken for {x.shape[0]} rows and this weight")
    prepared = isinstance(weight, LinearWeight)
    if prepared:
        weight, tiled, order, tile_rows = weight.rows, weight.tiled, weight.order, weight.tile_rows
    if isinstance(x, ScaledRows) and columns_on_16_bytes(x.rows):
        return skinny_gemm(x, weight, out_dtype or torch.bfloat16, tiled=tiled, order=order, tile_rows=tile_rows)
    columns = columns_on_16_bytes(x)      # (the product for few rows reads them where they lie, every other one takes a copy)
    if weight.dtype == torch.float32:
        return gemm_f32(x.contiguous() if columns else x, weight, None, out_dtype or x.dtype)
    if weight.dtype != torch.bfloat16 or x.dtype != torch.bfloat16:
        raise KernelError(f"linear: weight {weight.dtype} with activation {x.dtype} is not supported")
    if not columns:
        _check(x if not isinstance(x, ScaledRows) else x.rows, "x", (None, weight.shape[1]))
    elif x.shape[1] != weight.shape[1]:
        raise KernelError(f"x: shape {tuple(x.shape)}, expected {(None, weight.shape[1])}")
    _check(weight, "weight", (None, None))
    out_dtype = out_dtype or torch.bfloat16
    M, K = x.shape
    kind = _small_m_kernel(M, weight.shape[0], K, tiled is not None)
    if columns and kind != "skinny":
        x = x.contiguous()
    if prepared and M > SKINNY_MAX_M and (keep_slices or kind is None) and out_dtype == torch.bfloat16 and not torch.cuda.tunable.is_enabled():
        plan = few_tiles_plan(M, weight.shape[0], K, bool(keep_slices))
        if plan and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0 and weight.is_contiguous():
            return _by_plan(x, weight, plan, keep_slices)
    if kind == "skinny":
        ring = M >= RING_FEW_MIN_ROWS and ring_takes_few(x, LinearWeight(weight, tiled, order, tile_rows), keep_slices and out_dtype == torch.bfloat16)
        if ring:
            return ring_gemm(x, LinearWeight(weight, tiled, order, tile_rows), out_dtype, slices=0 if ring == 2 else 1, keep_slices=True)
        return skinny_gemm(x, weight, out_dtype, tiled=tiled, order=order, tile_rows=tile_rows)
    if kind == "wide":
        return wide_gemm(x, LinearWeight(weight, tiled, order, tile_rows), out_dtype, keep_slices=keep_slices)
    if kind == "staged":
        return staged_gemm(x, weight, out_dtype)
    if out_dtype == torch.float32:
        return torch.mm(x, weight.t(), out_dtype=torch.float32)
    if keep_slices and not torch.cuda.tunable.is_enabled():          # (where the library has timed its kernels its choice is the better one)
        plan = _tiles_sums_plan(M, weight.shape[0], K)
        if plan and torch.cuda.is_current_stream_capturing():
            plan = _tiles_sums_plan(M, weight.shape[0], K, True)
        if plan and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0:
            return _by_plan(x, weight, plan)
    if keep_slices:
        S = library_k_slices(M, weight.shape[0], K)
        if S > 1 and not torch.cuda.is_current_stream_capturing():
            # K cut into S slices as one batched product of the library with float32 results: [S, M, N] partial sums
            xs = x.view(M, S, K // S).transpose(0, 1)
            ws = weight.view(weight.shape[0], S, K // S).permute(1, 2, 0)
            return SliceSums(torch.bmm(xs, ws, out_dtype=torch.float32), out_dtype)
    return torch.matmul(x, weight.t())


def _by_plan(x: torch.Tensor, weight: torch.Tensor, plan: int, whole_in_float: bool = False):
    """The product that ``plan`` names; ``whole_in_float``: one slice stays a float sum, too, as the slices of the products that it is taken
    instead of are."""
    slices, tile, K = plan >> 8, plan & 255, x.shape[1]
    if slices > 1 or whole_in_float:
        return sums_tiles(x, weight, slices, -(-(-(-K // slices)) // 64) * 64, tile)
    return act_tiles(x, weight, ACT_NONE, tile)


FEW_MAX_ROWS = 2048              # rows, weight rows and k-values that ``few_tiles_plan`` was measured for
FEW_MIN_N, FEW_MAX_N, FEW_PAIRS_MAX_N = 256, 8192, 65536
FEW_MIN_K, FEW_MAX_K = 256, 20000
# products whose reader adds slices: k-values from which ..., multiplications up to which ..., against the library and against the product that shares x through LDS
FEW_SLICED = ((8192, 6.4e9, 3.2e9), (4096, 6.4e9, 1.6e9), (0, 3.2e9, 1.6e9))
FEW_WHOLE = ((512, 1, 1024), (1024, 1, 512), (3072, 128, 256))          # the plain product: k-values up to which ..., tiles of 64 x 64 from and up to which


@functools.lru_cache(maxsize=4096)
def few_tiles_plan(M: int, N: int, K: int, keep_slices: bool) -> int:
    """slices << 8 | tile of the tiles of ``gemm_tiles`` that take a model's weight [N, K] (a ``LinearWeight``) at 65 to 2,048 rows, 0: another product
    does.  Tiles of 64 x 64 and of 128 x 128 in three stages are made for these sizes, where tiles of 256 x 256 are few.  What the others take over
    their time, geometric mean and worst, 16,100 products of cold weights with what the slices cost their reader, by M N K:
        against the library's and large tiles', 129 rows on: up to 4e8 1.47 and 0.90, 4e8 to 1.6e9 1.6 and 0.72 (0.3 % below 0.97), 1.6e9 to 3.2e9 1.43 and
        0.71 (2 %), 3.2e9 to 6.4e9 with K of 4,096 to 8,192 1.15 and 0.82 (10 %), deeper 1.40 and 0.96; beyond the lines 3.2e9 to 6.4e9 with K up to 4,096 1.03
        and 0.66 (38 %), weights of more than 8,192 rows 0.79 to 0.9
        against the product that shares x through LDS, 65 to 128 rows: up to 8e8 1.7 and 1.09, 8e8 to 1.6e9 1.52 and 1.04, 1.6e9 to 3.2e9 with K from 8,192 on 1.40
        and 0.87 (8 %); beyond, with K of 4,096 to 8,192, 1.13 and 0.81 (30 %)
        in one slice (a float sum, as the slices are) 1.42, in more 1.60
    and, without slices, of 3,400 against the library: K up to 512 1.21 and 0.96, 512 to 1,024 1.16 and 0.84 (4 %; up to 512 tiles of 64 x 64: 18 to 24 % of more are
    slower), 1,024 to 3,072 with 128 to 256 tiles 1.11 and 0.89 (7 %), otherwise 1.05 with a third slower.  A bare tensor goes where ``_tiles_sums_plan`` says."""
    if not (SKINNY_MAX_M < M <= FEW_MAX_ROWS and FEW_MIN_N <= N <= FEW_MAX_N and FEW_MIN_K <= K <= FEW_MAX_K) or N % 8 or K % 8:
        return 0
    if keep_slices:
        _, most, most_streamed = next(line for line in FEW_SLICED if K >= line[0])
        if M * N * K > (most if M > WIDE_MAX_M else most_streamed):
            return 0
    else:
        tiles = -(-M // 64) * -(-N // 64)
        if not any(K <= deepest and least <= tiles < most for deepest, least, most in FEW_WHOLE):
            return 0
    return load_module("gemm_tiles").fn("ifx_gemm_tiles_few_plan", (I, I, I, I))(M, N, K, int(keep_slices))


@functools.lru_cache(maxsize=4096)
def _tiles_sums_plan(M: int, N: int, K: int, captured: bool = False) -> int:
    """slices << 8 | tile of a product by slices of tiles whose partial sums the caller adds (1: the plain product), 0: the library's.
    ``captured``: the call is being captured, so that its time on the host is none where it counts."""
    return load_module("gemm_tiles").fn("ifx_gemm_tiles_sums_plan", (I, I, I, I, I))(M, N, K, library_k_slices(M, N, K), int(captured))


LIBRARY_SLICE_MIN_K = 2048      # k-values a slice of a library product keeps at least
LIBRARY_MAX_SLICES = 8


@functools.lru_cache(maxsize=4096)
def library_k_slices(M: int, N: int, K: int) -> int:
    """Into how many slices of K a product that goes to the library is cut when the caller adds partial sums anyway.
    A product of many rows with a deep, narrow weight (down: 3,584 x 18,944) has few output tiles (the library's are
    about 256 x 256: 28 at 512 rows) and leaves most of the chip idle; cut into slices that still hold a few
    thousand k-values each, the same library fills it: at 512 rows 65 us instead of 124 (196 without tuning), at
    1,024 rows 112 instead of 188, at 2,048 rows 210 instead of 265.  A power of two, 1: not cut."""
    tiles = -(-M // 256) * -(-N // 256)
    S = 1
    while (2 * S <= LIBRARY_MAX_SLICES and 2 * S * tiles <= 256 and K % (16 * S) == 0
           and K // (2 * S) >= LIBRARY_SLICE_MIN_K):
        S *= 2
    return S


WIDE_FEW_ROWS_MIN_N = 16384               # rows of a weight (tall enough to fill the chip without slices of K) and ...
WIDE_FEW_ROWS_MIN_WEIGHT = 100_000_000    # ... its elements from which 9-16 rows take the product that shares x through LDS


def _tile_pairs_fit(N: int) -> bool:
    """Whether the product that splits K over a workgroup's waves takes the 16-row tiles of a weight of ``N`` rows in
    pairs (the rule of ifx_skinny_gemm: pairs halve its reads of x, and it takes them where they do not give the fullest
    of the 256 compute units more tiles than single tiles would)."""
    n_tiles = -(-N // 16)
    fullest = lambda nt: -(-(-(-n_tiles // nt)) // 256) * nt
    return -(-n_tiles // 2) >= 128 and fullest(2) <= fullest(1)


def _wide_for_few_rows(M: int, N: int, K: int) -> bool:
    """Whether up to 16 rows go to the product that shares x through LDS instead of the one that splits K over a
    workgroup's waves.  From 9 rows on the latter reads as much of x from the L2 as of W from memory; for large tall
    weights, which fill the chip without slices of K, the former then wins (both with the norm's factor per row; gate/up
    of the 7B shape at 9-16 rows 44.4 against 46.9 us, of the 14B shape 46 against 47-49, 32B 87 against 88-94 from 12
    rows, 72B 145 against 157-164; the heads of the 7B, 3B and 72B shapes from 12 rows: 177 against 185, 99 against 105
    and 385 against 414 at 16).  Where the other product cannot take tiles in pairs (gate/up of the 14B and 72B shapes)
    it reads x twice as often and loses from 6 rows on (14B 44.6 against 46.6-47.3 us at 6-8 rows, 72B 143-145 against
    146-149).  Smaller weights (gate/up of the 3B shape: 20 against 17 us) stay where they are."""
    if N < WIDE_FEW_ROWS_MIN_N:
        return _few_rows_in_slices(M, N, K)
    if N * K < WIDE_FEW_ROWS_MIN_WEIGHT:
        return False
    if M >= (12 if N >= 65536 else 9):
        return True
    return M >= 6 and N < 65536 and not _tile_pairs_fit(N)


UNEVEN_TILES_MIN_WEIGHT = 64_000_000      # elements from which a weight whose tiles lie unevenly on the chip is cut into slices of K


def _few_rows_in_slices(M: int, N: int, K: int) -> bool:
    """Whether 8-16 rows times a large weight of few rows go to the product that shares x through LDS and cuts K into slices
    (their sum left to the norm's kernel) instead of the one that adds into the stream itself.  The latter gives a
    workgroup whole row tiles: 5,120 rows are 320 tiles, two for 64 of the 256 compute units and one for the others,
    and the product takes as long as one of 8,192 rows (lower tiles do not help it: measured).  Slices of K fill the
    chip evenly whatever the number of tiles, at the price of the kernel that adds them (5.6 us).  down of the 32B shape
    (5,120 x 27,648) at 8 / 12 / 16 rows: 55 / 61 / 67 us against 43 + 5.6; of the 14B shape (5,120 x 13,824) 29 / 33 / 36
    against 24 + 5.6; its o (5,120 x 5,120: 14-17 against 11 + 5.6) is too small to gain, and weights whose tiles lie
    evenly (3,584 rows in tiles of 14, 8,192 rows) lose.  Decode steps: 8 requests at the 32B shape 13.4 -> 12.9 ms, 16 at
    the 14B shape 11.5 -> 11.3."""
    if M < (8 if N * K >= 2 * UNEVEN_TILES_MIN_WEIGHT else 9) or N * K < UNEVEN_TILES_MIN_WEIGHT:   # (8 rows: the smaller weight ties)
        return False
    tile_rows = choose_tile_rows(N)
    n_tiles = -(-N // tile_rows)
    return N < 0.7 * (-(-n_tiles // COMPUTE_UNITS) * COMPUTE_UNITS * tile_rows)


def _small_m_kernel(M: int, N: int, K: int, has_tiled: bool = False) -> Optional[str]:
    """Which of the streaming kernels takes a bfloat16 product of this shape, or None for the library.
    Measured on the 7B shapes: up to 16 rows the product that splits K over the waves of a workgroup (with x
    staged in LDS for very tall weights such as the head's when there is no tiled copy; 9-16 rows of large tall
    weights as from 17 rows, see _wide_for_few_rows); from 17 to 64 rows
    the product that shares x through LDS, which needs the tiled copy (without it, the first kernel up to 32
    rows on narrow weights); from 65 to 128 rows the same product for weights of few rows, whose K it cuts into
    slices to fill the chip where the library has too few output tiles to (down, o and q/k/v of the 7B shape:
    37-50, 15-21 and 16-22 us against 58-66, 30-34 and 30-37); beyond that, and for tall weights such as gate/up
    and the head, the library's tiles reuse the rows better.  (A model's weights go to small tiles first from 65 rows on where those
    are faster than either: ``few_tiles_plan``, ``few_pairs_take``.)"""
    if K % 8:
        return None
    if M <= 16:
        if has_tiled and _wide_for_few_rows(M, N, K):
            return "wide"
        return "staged" if N >= 65536 and not has_tiled else "skinny"
    if has_tiled and (M <= SKINNY_MAX_M or (M <= WIDE_MAX_M and N <= WIDE_MANY_ROWS_MAX_N)):
        return "wide"
    if M <= 32 and N <= 4096:
        return "skinny"
    return None


TILES_MAX_N = 1 << 22              # weight rows whose results a buffer's offsets reach (128 rows of them, 2 bytes each)
MANY_TILES_MIN_ROWS = 129          # (up to 128 rows are mostly the streaming products')
# k-values up to which ...: the least M N / 65,536 (tiles of 256 x 256) from which ..., of gate/up pairs and of products without a gate
MANY_TILES = ((800, 16, 32), (1536, 32, 48), (2560, 96, 96), (4096, 128, 128))


def many_tiles_take(M: int, N: int, K: int, gated: bool = True) -> bool:
    """Whether the product for many rows with the activation as its epilogue takes a bfloat16 weight [N, K] because its tiles fill the
    chip.  1,450 sizes drawn over 129 to 8,192 rows, 16 to 61,000 weight rows, 8 to 4,096 k-values, cold weights, the library's product and
    the activation's launch in the time of this one, geometric mean and worst, gate/up (silu) : without a gate (gelu):
        K      up to 800: 16 to 32 tiles 1.28 to 1.51, 1.15 : 0.92, 0.77     32 to 64 1.47 to 1.86, 1.24 : 1.06 to 1.25, 0.92
                          more 1.66 to 2.2, 1.33 : 1.46 to 1.69, 1.20
        K 800 to 1,536:   32 to 48 1.31, 1.11 : 0.95, 0.79     more 1.45, 1.08 : 1.34, 1.03
        K 1,536 to 2,560: up to 64 0.90, 0.59 : 0.70, 0.46     64 to 96 1.11, 0.82 : 1.12, 0.92     more 1.30, 0.90 : 1.22, 0.85
        K 2,560 to 4,096: up to 64 0.78, 0.53 : 0.68, 0.38     64 to 96 0.95, 0.90 : 1.02, 0.93     more 1.27, 1.00 : 1.23, 0.96
    (of 4,096 to 8,192 k-values, warm weights: 128 to 256 tiles 1.06 and 0.76, more 1.11 and 0.94; there the library keeps the product).
    Where the library has timed its kernels the lines are the same (42 sizes beyond them: 1.33 and 0.97)."""
    if M < MANY_TILES_MIN_ROWS or K < 64 or K % 8 or N % (16 if gated else 8) or N > TILES_MAX_N:
        return False
    return any(K <= deepest and M * N >= 65536 * (pairs if gated else plain) for deepest, pairs, plain in MANY_TILES)


FEW_TILES = ((192, 0), (400, 4), (600, 8), (1536, 24))          # the same of gate/up pairs whose tiles do not fill it


def pairs_tiles_take(M: int, N: int, K: int) -> bool:
    """Whether that product takes gate/up pairs [N, K] of shallow weights also where its tiles do not fill the chip, for the launch that it
    saves: measured as for ``many_tiles_take``, geometric mean and worst
        K up to 192: up to 4 tiles 1.33, 0.97, more 1.20, 1.03     192 to 400: up to 4 1.17, 0.91 (a quarter of them slower), more 1.19, 0.98
        400 to 600: up to 8 1.04, 0.78, more 1.16, 1.10     600 to 800: 0.97, 0.71     800 to 1,536: up to 24 0.86, 0.57, more 1.14, 1.08.
    Where the caller has the library time its kernels (``enable_library_gemm_tuning``), its choice is the faster one at such sizes."""
    if M < MANY_TILES_MIN_ROWS or N % 4 or N > TILES_MAX_N or K % 8 or K > FEW_TILES[-1][0]:
        return False
    return any(K <= deepest and M * N >= 65536 * tiles for deepest, tiles in FEW_TILES) and not torch.cuda.tunable.is_enabled()


def few_pairs_take(M: int, N: int, K: int) -> bool:
    """Whether that product takes a model's gate/up pairs [N, K] (a ``LinearWeight``) at 65 to 2,048 rows, where tiles by small waves are among its
    choices.  The library's product and the activation, or up to 128 rows the product that shares x through LDS, over this one's time, geometric mean
    and worst of 8,700: up to 128 rows 2.0 and 0.88; more, K up to 1,536 and 16 tiles of 256 x 256 1.46 and 0.94 (beyond, ``many_tiles_take`` has most of them
    anyway), 1,536 to 2,560 and up to 64 tiles 1.29 and 0.87, 2,560 to 4,096 and 2 to 16 tiles 1.24 and 0.78 (3 % below 0.97; fewer 0.96 and 0.83); 1,536 to 2,560
    and more tiles 1.0, from 700 rows on 0.98 and 0.88."""
    if not (SKINNY_MAX_M < M <= FEW_MAX_ROWS and FEW_MIN_N <= N <= FEW_PAIRS_MAX_N and N % 4 == 0 and FEW_MIN_K <= K <= 4096 and K % 8 == 0):
        return False
    tiles = M * N / 65536
    fits = K <= 1536 or (M <= 300 or tiles <= 64 if K <= 2560 else (M <= WIDE_MAX_M or tiles >= 2) and tiles <= 16)
    return fits and not torch.cuda.tunable.is_enabled()


def swiglu_tiles(x: torch.Tensor, pairs: torch.Tensor, act: int = ACT_SILU, limit: float = 0.0, tile: int = -1) -> torch.Tensor:
    """``linear_swiglu`` of many rows in bfloat16 as one launch ([N, K] ``pairs``, N a multiple of 4 and K of 8, both on 16 bytes);
    ``tile``: one of the kernel's tiles instead of its choice."""
    _check(pairs, "weight_pairs", (None, None), torch.bfloat16)
    N, K = pairs.shape
    _check(x, "x", (None, K), torch.bfloat16)
    out = empty((x.shape[0], N // 2), torch.bfloat16, x)
    _call(load_module("gemm_tiles"), "ifx_gemm_tiles", _TILES_ARGS, x, pairs, out,
          x.shape[0], N, K, 0, int(act), float(limit), int(tile), _stream())
    return out


def act_tiles(x: torch.Tensor, weight: torch.Tensor, act: int, tile: int = -1) -> torch.Tensor:
    """``linear_act`` of many rows in bfloat16 as one launch ([N, K] ``weight``, N even and K a multiple of 8, both on 16 bytes);
    ``tile`` as for ``swiglu_tiles``, but not 2."""
    _check(weight, "weight", (None, None), torch.bfloat16)
    N, K = weight.shape
    _check(x, "x", (None, K), torch.bfloat16)
    out = empty((x.shape[0], N), torch.bfloat16, x)
    _call(load_module("gemm_tiles"), "ifx_gemm_tiles", _TILES_ARGS, x, weight, out,
          x.shape[0], N, K, 1, int(act), 0.0, int(tile), _stream())
    return out


def sums_tiles(x: torch.Tensor, weight: torch.Tensor, slices: int, slice_k: int, tile: int) -> "SliceSums":
    """bfloat16 x [M, K] times ``weight`` [N, K] transposed as ``SliceSums`` over ``slices`` of ``slice_k`` values of K (a multiple of
    64), N a multiple of 4, K of 8, both on 16 bytes; ``tile``: one of the kernel's tiles but 2."""
    _check(weight, "weight", (None, None), torch.bfloat16)
    N, K = weight.shape
    _check(x, "x", (None, K), torch.bfloat16)
    parts = empty((slices, x.shape[0], N), torch.float32, x)
    _call(load_module("gemm_tiles"), "ifx_gemm_tiles_sums", (P, P, P, I, I, I, I, I, I, P), x, weight, parts,
          x.shape[0], N, K, int(slices), int(slice_k), int(tile), _stream())
    return SliceSums(parts, torch.bfloat16)


_TILES_ARGS = (P, P, P, I, I, I, I, I, F, I, P)


def linear_swiglu(x: torch.Tensor, weight_pairs, act: int = ACT_SILU, limit: float = 0.0) -> torch.Tensor:
    """act(x Wg^T) * (x Wu^T) (``act``: ACT_SILU, ACT_GELU_TANH, or ACT_CLAMPED_SWISH with its ``limit``) where ``weight_pairs``
    [2I, K] (a tensor or a ``LinearWeight``) alternates the rows of Wg and Wu; ``x`` as for ``linear``.  For few rows (not with ACT_CLAMPED_SWISH) and
    for many (``pairs_tiles_take``, ``many_tiles_take``) the activation is the product's epilogue; otherwise a second kernel applies it."""
    M, K = x.shape
    if isinstance(x, ScaledRows) and not takes_scaled_rows(M, weight_pairs):
        raise KernelError(f"linear_swiglu: scaled rows are not taken for {M} rows and this weight")
    rows, tiled, tile_rows = ((weight_pairs.rows, weight_pairs.tiled, weight_pairs.tile_rows) if isinstance(weight_pairs, LinearWeight)
                              else (weight_pairs, None, 16))
    if isinstance(weight_pairs, LinearWeight) and weight_pairs.order is not None:
        raise KernelError("linear_swiglu: a tile order is not supported for gate/up pairs")
    columns = columns_on_16_bytes(x)          # (as for ``linear``)
    if not isinstance(x, ScaledRows) and rows.dtype == torch.bfloat16 and x.dtype == torch.bfloat16 and K == rows.shape[1] \
            and (pairs_tiles_take(M, rows.shape[0], K) or many_tiles_take(M, rows.shape[0], K)
                 or isinstance(weight_pairs, LinearWeight) and few_pairs_take(M, rows.shape[0], K)):
        whole = x.contiguous() if columns else x
        if whole.data_ptr() % 16 == 0 and rows.is_contiguous() and rows.data_ptr() % 16 == 0:
            return swiglu_tiles(whole, rows, act, limit)
    if rows.dtype == torch.float32 and x.dtype == torch.float32 and not isinstance(x, ScaledRows):
        return gemm_f32(x.contiguous() if columns else x, rows, gated=act, limit=limit)
    if act == ACT_CLAMPED_SWISH:
        return swiglu(linear(x, weight_pairs), interleaved=True, act=act, limit=limit)
    if rows.dtype == torch.bfloat16 and x.dtype == torch.bfloat16:
        kind = _small_m_kernel(M, rows.shape[0], K, tiled is not None)
        if kind == "skinny":
            if ring_takes_few(x, weight_pairs) and rows.shape[0] % 2 == 0:
                return ring_gemm(x, weight_pairs, swiglu_pairs=True, act=act)
            return skinny_gemm(x, rows, torch.bfloat16, swiglu_pairs=True, tiled=tiled, tile_rows=tile_rows, act=act)
        if columns:
            x = x.contiguous()
        if kind == "wide":
            return wide_gemm(x, weight_pairs, torch.bfloat16, swiglu_pairs=True, act=act)
        if kind == "staged":
            return staged_gemm(x, rows, torch.bfloat16, swiglu_pairs=True, act=act)
    return swiglu(linear(x, rows), interleaved=True, act=act)


# ----------------------------------------------------------------------------------------
def attention_plain(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, row_req: torch.Tensor,
                    positions: torch.Tensor, block_table: torch.Tensor, window: Optional[int],
                    scale: float, keep_first: int = 0, sink: Optional[float] = None,
                    gate: Optional[torch.Tensor] = None, sinks: Optional[torch.Tensor] = None, chunk: Optional[int] = None,
                    differential: Optional[Tuple[float, float, float]] = None, row_waves: int = 0,
                    rows: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal (optionally windowed) attention of q [T, nH, d] over the paged cache (K [pages, nKV, page, d],
    V [pages, nKV, dv, page]; dv may differ from d); returns [T, nH*dv].  ``keep_first``: a windowed query also sees
    the first so many positions of its request; ``sink``: the score of a key without value that is added to the
    softmax's denominator (None: no such key), ``sinks`` float32 [nH]: such a score for every head; ``gate`` float32
    [T, nH]: a factor on every head's output; ``chunk``: a query sees only keys of its own block of that many positions,
    counted from the sequence's start.  ``differential`` (lambda, out_scale, eps): q and the keys hold two vectors of
    d / 2 elements per head, each pair a softmax map of its own over the same values; a head's output is map 1 minus
    lambda times map 2, divided by its root mean square (eps inside the root), times out_scale.  ``row_waves``: waves to a row and
    head, 1 or 4 (0 lets the kernel choose; the same bits either way).  ``rows`` int32: only these rows of ``out`` are written."""
    _check(q, "q", (None, None, None))
    T, nH, d = q.shape
    maps = 2 if differential is not None else 1
    if d % maps:
        raise KernelError(f"attention_plain: two maps need an even row, got {d}")
    lam, out_scale, norm_eps = differential if differential is not None else (0.0, 1.0, 0.0)
    if sinks is not None:
        _check(sinks, "sinks", (nH,), torch.float32)
    _check(k_cache, "k_cache", (None, None, None, d), q.dtype)
    n_pages, nKV, page_size, _ = k_cache.shape
    _check(v_cache, "v_cache", (n_pages, nKV, None, page_size), q.dtype)
    dv = v_cache.shape[2]
    _check(row_req, "row_req", (T,), torch.int32)
    _check(positions, "positions", (T,), torch.int32)
    _check(block_table, "block_table", (None, None), torch.int32)
    if gate is not None:
        _check(gate, "gate", (T, nH), torch.float32)
    if out is None:
        out = empty((T, nH * dv), q.dtype, q)
    else:
        _check(out, "out", (T, nH * dv), q.dtype)
    if rows is not None:
        _check(rows, "rows", (None,), torch.int32)
        T = rows.shape[0]
    _call(load_module("attn_plain"), "ifx_attn_plain", (P, P, P, P, I, P, P, P, I, I, I, I, I, I, I, I, F, I, I, F, P, P, I, I, F, F, F, I, P, P),
          q, k_cache, v_cache, out, _dt(q), row_req,
          positions, block_table, block_table.shape[1], T, nH, nKV, d // maps, dv, page_size,
          int(window or 0), float(scale), int(keep_first or 0), 0 if sink is None else 1, float(sink or 0.0), gate,
          sinks, int(chunk or 0), maps, float(lam), float(out_scale), float(norm_eps), int(row_waves), rows, _stream())
    return out


@functools.lru_cache(maxsize=None)
def _attention_f32_cols(d: int, dv: int, maps: int, page_size: int) -> int:
    return load_module("attn_f32").fn("ifx_attn_f32_cols", (I, I, I, I))(d, dv, maps, page_size)


def attention_f32_cols(dtype: torch.dtype, d: int, dv: int, maps: int, page_size: int) -> int:
    """(row, query head) pairs to a workgroup of ``attention_f32`` for keys of ``maps`` vectors of ``d`` elements and values of ``dv``;
    0: it has no kernel for them."""
    return _attention_f32_cols(d, dv, maps, page_size) if dtype == torch.float32 else 0


def attention_f32(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, out: torch.Tensor, tiles: torch.Tensor,
                  q_start: torch.Tensor, q_len: torch.Tensor, kv_len: torch.Tensor, block_table: torch.Tensor, window: Optional[int],
                  scale: float, keep_first: int = 0, sink: Optional[float] = None, gate: Optional[torch.Tensor] = None,
                  sinks: Optional[torch.Tensor] = None, chunk: Optional[int] = None,
                  differential: Optional[Tuple[float, float, float]] = None, split: bool = False) -> None:
    """What ``attention_plain`` computes, the same bits, for whole tiles of rows in 32 bits on the matrix cores: ``tiles`` int32 [n, 2]
    (request, first of ``attention_f32_cols`` columns; the columns of a request are its rows in this step times the query heads
    of a kv head, and the first must lie among them).  Rows of requests without tiles stay as they are in ``out``.
    ``split``: the four parts of a row's keys by workgroups of their own (the same bits)."""
    _check(q, "q", (None, None, None), torch.float32)
    T, nH, d = q.shape
    maps = 2 if differential is not None else 1
    if d % maps:
        raise KernelError(f"attention_f32: two maps need an even row, got {d}")
    lam, out_scale, norm_eps = differential if differential is not None else (0.0, 1.0, 0.0)
    if sinks is not None:
        _check(sinks, "sinks", (nH,), torch.float32)
    _check(k_cache, "k_cache", (None, None, None, d), torch.float32)
    n_pages, nKV, page_size, _ = k_cache.shape
    _check(v_cache, "v_cache", (n_pages, nKV, None, page_size), torch.float32)
    dv = v_cache.shape[2]
    _check(out, "out", (T, nH * dv), torch.float32)
    _check(tiles, "tiles", (None, 2), torch.int32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (kv_len, "kv_len")):
        _check(t, nm, (R,), torch.int32)
    _check(block_table, "block_table", (R, None), torch.int32)
    if gate is not None:
        _check(gate, "gate", (T, nH), torch.float32)
    part_o = part_ml = None
    if split or maps > 1:
        part_o, part_ml = (empty((T, nH, maps, 4 if split else 1, n), torch.float32, q) for n in (dv, 2))
    _call(load_module("attn_f32"), "ifx_attn_f32", (P, P, P, P, P, I, P, P, P, P, I, I, I, I, I, I, I, F, I, I, F, P, P, I, I, F, F, F, I, P, P, P),
          q, k_cache, v_cache, out, tiles, tiles.shape[0], q_start, q_len, kv_len, block_table, block_table.shape[1], nH, nKV, d // maps,
          dv, page_size, int(window or 0), float(scale), int(keep_first or 0), 0 if sink is None else 1, float(sink or 0.0), gate,
          sinks, int(chunk or 0), maps, float(lam), float(out_scale), float(norm_eps), int(split), part_o, part_ml, _stream())


# ----------------------------------------------------------------------------------------
DELTA_THREAD_CHANNELS = (4, 8, 16, 32, 64)  # key channels of a column of S a thread may hold
DELTA_MAX_PADDED_DIM, DELTA_MAX_COLS, DELTA_THREADS = 256, 128, 256
# ... at most this many in steps of single tokens that ``delta_step`` does not take (64 decoded rows, us with 4, 8 and 16: 16 heads of 64 x 128 in 32 bits 84.9, 51.0,
DELTA_DECODE_MAX_CHANNELS = 8               # 58.5, 4 heads of 128 x 256 in bfloat16 110.7, 71.2, 79.6)


def delta_padded_dim(d: int) -> int:
    """The key channels of a head padded to a power of two (at least 4): what a column of S takes in a request's state."""
    p = 4
    while p < d:
        p *= 2
    if p > DELTA_MAX_PADDED_DIM:
        raise KernelError(f"delta rule: heads of {d} key channels (at most {DELTA_MAX_PADDED_DIM})")
    return p


def delta_layout(d: int, dv: int, single_tokens: bool = False) -> Tuple[int, int, int]:
    """(channels a thread, threads a column, columns a workgroup) of the delta rule's kernel for heads of ``d`` key channels
    and ``dv`` values.  The threads of a column are a power of two of neighbouring lanes that share the padded channels; a
    workgroup has up to 256 threads and a head's columns are dealt to as many workgroups as that takes.  The state's layout
    does not depend on the choice, so a step takes the one that suits it: a prompt's portion is a chain from token to token,
    which is shortest with the fewest channels a thread; steps of single tokens are many short workgroups, of which there
    should be few (``single_tokens``)."""
    dpad = delta_padded_dim(d)
    found = []
    for ch in DELTA_THREAD_CHANNELS:
        if ch > dpad or dpad // ch > 64:
            continue
        ks = dpad // ch
        cols = max(1, min(dv, DELTA_THREADS // ks, DELTA_MAX_COLS))
        threads = -(-cols * ks // 64) * 64
        if dpad <= threads and 2 * cols <= threads:         # (each thread fetches its share of a stage of sixteen tokens)
            found.append((ch, ks, cols))
    if not found:
        raise KernelError(f"delta rule: heads of {d} key channels and {dv} values fit no layout of the kernel")
    if single_tokens:
        few = [f for f in found if f[0] <= DELTA_DECODE_MAX_CHANNELS] or found
        return min(few, key=lambda f: (-(-dv // f[2]), f[0]))
    return found[0]


def delta_state_floats(n_heads: int, d: int, dv: int) -> int:
    delta_layout(d, dv)
    return n_heads * dv * delta_padded_dim(d)


def delta_rule(u: torch.Tensor, rows: torch.Tensor, cols: Tuple[int, int, int], A_log: torch.Tensor, dt_bias: torch.Tensor,
               norm_w: torch.Tensor, eps: float, n_heads: int, n_kv_heads: int, d: int, dv: int, state: torch.Tensor,
               state_offset: int, q_start: torch.Tensor, q_len: torch.Tensor, slots: torch.Tensor,
               single_tokens: bool = False) -> torch.Tensor:
    """The gated delta rule over a step's rows (see csrc/delta.hip).  ``u`` [T, >= 2 G d + H dv] holds per row the q heads,
    the k heads and the v heads (after their convolution), ``rows`` [T, ld] the gate's H dv columns from ``cols[0]``, beta's
    H from ``cols[1]`` and the decay's H from ``cols[2]``, both in the activation type.  ``A_log``, ``dt_bias`` float32 [H],
    ``norm_w`` [dv].  A request's S lies ``state_offset`` floats into its row of ``state`` [slots, n] (float32), zero for a
    request that starts.  ``single_tokens``: every request brings one row (the launch then takes few, larger workgroups).
    Returns [T, H dv] in u's type."""
    _check(u, "u", (None, None))
    T, ldu = u.shape
    _check(rows, "rows", (T, None), u.dtype)
    ldr = rows.shape[1]
    H, G = n_heads, n_kv_heads
    col_g, col_b, col_a = cols
    if ldu < 2 * G * d + H * dv or col_g + H * dv > ldr or col_b + H > ldr or col_a + H > ldr:
        raise KernelError("delta_rule: the rows are narrower than the columns named")
    _check(A_log, "A_log", (H,), torch.float32)
    _check(dt_bias, "dt_bias", (H,), torch.float32)
    _check(norm_w, "norm_w", (dv,))
    _check(state, "state", (None, None), torch.float32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    ch, ks, cols = delta_layout(d, dv, single_tokens)
    if state_offset + H * dv * ch * ks > state.shape[1]:
        raise KernelError("delta_rule: the state rows are too short")
    out = empty((T, H * dv), u.dtype, u)
    o_raw = empty((T, H * dv), torch.float32, u)
    _call(load_module("delta"), "ifx_delta_rule", (P, I, P, I, I, I, I, I, P, P, P, I, F, P, LL, LL, P, P, P, P, P, I, I, I, I, I, I, I, I, I, P),
          u, ldu, rows, ldr, col_g, col_b, col_a, _dt(u), A_log, dt_bias,
          norm_w, _dt(norm_w), float(eps), state, state.shape[1], int(state_offset), q_start,
          q_len, slots, out, o_raw, T, R, H, G, d, dv, ch, ks, cols, _stream())
    return out


DELTA_STEP_TAPS = 4         # ... of the convolution that ``delta_step`` takes along


def delta_step_takes(dtype: torch.dtype, d: int, dv: int, state_offset: int, state: torch.Tensor) -> bool:
    """Whether ``delta_step`` takes single tokens of these heads."""
    return (dtype == torch.bfloat16 and state_offset % 4 == 0 and state.shape[1] % 4 == 0
            and bool(load_module("delta").fn("ifx_delta_step_takes", (I, I))(delta_padded_dim(d), dv)))


def delta_step(u: torch.Tensor, conv_w: Optional[torch.Tensor], rows: torch.Tensor, cols: Tuple[int, int, int], A_log: torch.Tensor,
               dt_bias: torch.Tensor, norm_w: torch.Tensor, eps: float, n_heads: int, n_kv_heads: int, d: int, dv: int, state: torch.Tensor,
               state_offset: int, q_start: torch.Tensor, q_len: torch.Tensor, slots: torch.Tensor) -> torch.Tensor:
    """``delta_rule`` of a step of single tokens in bfloat16 as one launch (``delta_step_takes``), and with ``conv_w`` [2 G d + H dv,
    DELTA_STEP_TAPS] (as many q and k heads as heads) ``causal_conv_silu`` of the first so many columns of ``u`` before it, whose state begins a
    request's row.  What lies between the two, and between the walk and its norm, is not rounded."""
    _check(u, "u", (None, None), torch.bfloat16)
    T, ldu = u.shape
    _check(rows, "rows", (T, None), torch.bfloat16)
    H, G = n_heads, n_kv_heads
    channels = 2 * G * d + H * dv
    col_g, col_b, col_a = cols
    if ldu < channels or col_g + H * dv > rows.shape[1] or max(col_b, col_a) + H > rows.shape[1]:
        raise KernelError("delta_step: the rows are narrower than the columns named")
    if conv_w is not None:
        _check(conv_w, "conv_w", (channels, DELTA_STEP_TAPS))
    _check(A_log, "A_log", (H,), torch.float32)
    _check(dt_bias, "dt_bias", (H,), torch.float32)
    _check(norm_w, "norm_w", (dv,))
    _check(state, "state", (None, None), torch.float32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    out = empty((T, H * dv), u.dtype, u)
    _call(load_module("delta"), "ifx_delta_step", (P, I, P, I, I, P, I, I, I, I, P, P, P, I, F, P, LL, LL, P, P, P, P, I, I, I, I, I, I, I, P),
          u, ldu, conv_w, DT_F32 if conv_w is None else _dt(conv_w), 0 if conv_w is None else DELTA_STEP_TAPS, rows, rows.shape[1], col_g, col_b, col_a,
          A_log, dt_bias, norm_w, _dt(norm_w), float(eps), state, state.shape[1], int(state_offset), q_start, q_len, slots, out, T, R, H, G, d, dv,
          delta_padded_dim(d), _stream())
    return out


def diff_expand(q: torch.Tensor) -> torch.Tensor:
    """q [T, H, 2 d] -> [T, 2 H, 2 d]: head 2 h is [q1 | 0], head 2 h + 1 is [0 | q2] (the two maps of differential attention as
    heads of their own against keys whose rows hold both maps' vectors)."""
    _check(q, "q", (None, None, None))
    T, H, two_d = q.shape
    if two_d % 2:
        raise KernelError("diff_expand: a row of two maps has an even number of elements")
    out = empty((T, 2 * H, two_d), q.dtype, q)
    _call(load_module("rowwise"), "ifx_diff_expand", (P, P, I, LL, I, P), q, out, _dt(q), T * H, two_d // 2, _stream())
    return out


def diff_combine(a, n_heads: int, dv: int, lam: float, out_scale: float, eps: float) -> torch.Tensor:
    """a [T, 2 H dv] (per head the two maps' outputs, one after the other; also ``SplitRows``) -> [T, H dv]: o =
    a1 - lam a2, divided by its root mean square over dv (eps inside the root), times out_scale."""
    if isinstance(a, SplitRows):
        if a.n_heads != 2 * n_heads or a.width != dv or a.sinks is not None:
            raise KernelError(f"diff_combine: splits of {a.n_heads} heads of {a.width} where two maps of {n_heads} of {dv} are joined")
        out = empty((a.shape[0], n_heads * dv), a.dtype, a.part_o)
        _call(load_module("rowwise"), "ifx_diff_combine_splits", (P, P, I, P, I, I, I, F, F, F, P), a.part_o, a.part_ml, a.n_splits, out, a.shape[0],
              n_heads, dv, float(lam), float(out_scale), float(eps), _stream())
        return out
    _check(a, "a", (None, 2 * n_heads * dv))
    T = a.shape[0]
    out = empty((T, n_heads * dv), a.dtype, a)
    _call(load_module("rowwise"), "ifx_diff_combine", (P, P, I, LL, I, F, F, F, P), a, out, _dt(a), T * n_heads, dv,
          float(lam), float(out_scale), float(eps), _stream())
    return out


def stream_add(stream: torch.Tensor, rows: Optional[torch.Tensor] = None, vec: Optional[torch.Tensor] = None) -> torch.Tensor:
    """stream [T, H] (float32) += rows [T, H] (float32) + vec [H], in place; either operand may be None."""
    _check(stream, "stream", (None, None), torch.float32)
    T, H = stream.shape
    if rows is not None:
        _check(rows, "rows", (T, H), torch.float32)
    if vec is not None:
        _check(vec, "vec", (H,))
    _call(load_module("rowwise"), "ifx_stream_add", (P, P, P, I, I, I, P), stream, rows, vec,
          _dt(vec) if vec is not None else 0, T, H, _stream())
    return stream


# ----------------------------------------------------------------------------------------
def causal_conv_silu(x: torch.Tensor, channels: int, weight: torch.Tensor, bias: Optional[torch.Tensor], state: torch.Tensor,
                     row_req: torch.Tensor, q_start: torch.Tensor, q_len: torch.Tensor, slots: torch.Tensor) -> torch.Tensor:
    """silu of a causal convolution per channel over each request's rows: the first ``channels`` columns of ``x``
    [T, >= channels] with ``weight`` [channels, taps] (the last column is the current token's) and ``bias``.  A request's
    last taps - 1 inputs live in the first channels * (taps - 1) floats of its row of ``state`` [slots, n] (float32,
    zero for a request that starts), are read as the inputs before this step's and replaced by this step's last.
    ``row_req`` [T], ``q_start`` / ``q_len`` / ``slots`` [R] (int32) describe the step.  Returns [T, channels]."""
    _check(x, "x", (None, None))
    T, ld = x.shape
    _check(weight, "weight", (channels, None))
    taps = weight.shape[1]
    if bias is not None:
        _check(bias, "bias", (channels,), weight.dtype)
    _check(state, "state", (None, None), torch.float32)
    _check(row_req, "row_req", (T,), torch.int32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    out = empty((T, channels), x.dtype, x)
    _call(load_module("ssm"), "ifx_causal_conv", (P, I, I, P, P, I, P, LL, P, P, P, P, P, I, I, I, I, P),
          x, _dt(x), ld, weight, bias, _dt(weight), state, state.shape[1],
          row_req, q_start, q_len, slots, out, T, R, channels, taps, _stream())
    return out


def selective_scan(u: torch.Tensor, dt_raw: torch.Tensor, dt_bias: torch.Tensor, A: torch.Tensor, bc: torch.Tensor,
                   D: torch.Tensor, z: torch.Tensor, state: torch.Tensor, state_offset: int, q_start: torch.Tensor,
                   q_len: torch.Tensor, slots: torch.Tensor, chunks: Optional[Dict[str, object]] = None) -> torch.Tensor:
    """The recurrence of a selective state-space mixer over each request's rows, then the gate:
    dt = softplus(dt_raw + dt_bias); S[c, n] <- exp(dt A[c, n]) S[c, n] + dt u[c] B[n]; y[c] = sum_n S[c, n] C[n] + D[c] u[c];
    out = y * silu(z).  ``u`` [T, C], ``dt_raw`` float32 [T, C], ``A`` float32 [C, N] (negative), ``bc`` [T, >= 2N] with B
    then C, ``z`` a view [T, C] of rows that may be wider (its row stride is taken), ``state`` float32 [slots, n] with a
    request's S at ``state_offset`` of its row.  All of the recurrence is float.  Returns [T, C] in u's type.

    ``chunks`` (from ``scan_chunks``): the requests' rows cut into chunks that run side by side, each first from a zero
    state, then from the state that the chunks before it leave (the recurrence is linear in S); the same function up to
    the rounding of float sums taken in another order."""
    _check(u, "u", (None, None))
    T, C = u.shape
    _check(dt_raw, "dt_raw", (T, C), torch.float32)
    _check(A, "A", (C, None), torch.float32)
    N = A.shape[1]
    _check(dt_bias, "dt_bias", (C,))
    _check(D, "D", (C,), dt_bias.dtype)
    _check(bc, "bc", (T, None), u.dtype)
    if not (isinstance(z, torch.Tensor) and z.is_cuda and z.dtype == u.dtype and tuple(z.shape) == (T, C) and z.stride(1) == 1):
        raise KernelError("selective_scan: z must be a [T, C] view with contiguous rows in u's type")
    _check(state, "state", (None, None), torch.float32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    out = empty((T, C), u.dtype, u)
    n_chunks, max_chunk, lists = 0, 0, (0, 0, 0, 0, 0, 0)
    if chunks is not None:
        n_chunks, max_chunk = chunks["req"].shape[0], int(chunks["rows"])
        for nm in ("req", "t0", "len"):
            _check(chunks[nm], f"chunks.{nm}", (n_chunks,), torch.int32)
        _check(chunks["req_chunk0"], "chunks.req_chunk0", (R + 1,), torch.int32)
        chunk_state = empty((n_chunks, C, N), torch.float32, u)
        chunk_dt = empty((n_chunks, C), torch.float32, u)
        lists = (chunks["req"].data_ptr(), chunks["t0"].data_ptr(), chunks["len"].data_ptr(), chunks["req_chunk0"].data_ptr(),
                 chunk_state.data_ptr(), chunk_dt.data_ptr())
    _call(load_module("ssm"), "ifx_selective_scan",
          (P, I, P, P, P, P, I, P, I, P, I, P, LL, LL, P, P, P, P, I, I, I, I, I, I, P, P, P, P, P, P, P),
          u, _dt(u), dt_raw, dt_bias, A, bc, bc.shape[1], D,
          _dt(D), z, z.stride(0) if T else C, state, state.shape[1], int(state_offset), q_start,
          q_len, slots, out, T, R, C, N, n_chunks, max_chunk, *lists, _stream())
    return out


def scan_chunks(q_start, q_len, chunk: int, device) -> Dict[str, object]:
    """The lists ``selective_scan`` takes as ``chunks``: every request's rows (host arrays ``q_start`` / ``q_len`` of the
    step) cut into chunks of up to ``chunk`` rows, in one upload."""
    import numpy as np
    req, t0, ln, first = [], [], [], [0]
    for r, (s0, n) in enumerate(zip(q_start.tolist(), q_len.tolist())):
        for at in range(0, n, chunk):
            req.append(r); t0.append(s0 + at); ln.append(min(chunk, n - at))
        first.append(len(req))
    n = len(req)
    pad = lambda v: v + [0] * (-len(v) % 4)
    packed = upload(np.asarray(pad(req) + pad(t0) + pad(ln) + first, dtype=np.int32), device)
    w = n + -n % 4
    return {"req": packed[:n], "t0": packed[w:w + n], "len": packed[2 * w:2 * w + n], "req_chunk0": packed[3 * w:3 * w + len(first)],
            "rows": int(chunk)}       # (the most rows a chunk has: the kernels keep a chunk's B and C in LDS)


# ----------------------------------------------------------------------------------------
GLA_THREAD_CHANNELS = ((16, 512), (32, 1024), (64, 512), (128, 256))   # channels of S a thread may hold, and the threads a workgroup may then have


def gla_layout(d: int, dv: int) -> Tuple[int, int]:
    """(channels a thread holds, threads per column) for a head of d key channels and dv values: the first pairing whose
    workgroup (dv columns times the threads of a column) fits; failing that, the first in which a thread holds several
    columns (4 with 16 channels, 2 with 32: what its registers take).  A request's S takes heads * dv * parts * channels
    floats."""
    def parts_for(dp):
        parts = 1
        while parts * dp < d:
            parts *= 2
        return parts
    for dp, max_threads in GLA_THREAD_CHANNELS:
        parts = parts_for(dp)
        if parts <= 64 and max(dv * parts, d) <= max_threads:     # (a thread per key channel loads a stage's q, k and decays)
            return dp, parts
    for dp, cols in ((16, 4), (32, 2)):
        parts = parts_for(dp)
        if parts <= 64 and max(-(-dv // cols) * parts, d) <= 1024:
            return dp, parts
    raise KernelError(f"gla: a head of {d} key channels and {dv} values does not fit a workgroup")


def gla_takes_blocks(rows: torch.Tensor, cols: Tuple[int, int, int, int], z: torch.Tensor, z_bias: Optional[torch.Tensor], d: int, dv: int) -> bool:
    """Whether ``gla_scan`` runs these rows' chunks on the matrix cores: bfloat16, heads of the layout for 64 key channels and 128 values, everything it reads on
    16 bytes (the rule of blocks_take in csrc/gla.hip)."""
    dp, parts = gla_layout(d, dv)
    return (rows.dtype == torch.bfloat16 and dp * parts == 64 and d % 4 == 0 and dv == 128 and rows.shape[1] % 8 == 0
            and all((rows.data_ptr() + 2 * c) % 16 == 0 for c in cols) and z.data_ptr() % 16 == 0 and (z_bias is None or z_bias.data_ptr() % 16 == 0))


def gla_state_floats(n_heads: int, d: int, dv: int) -> int:
    dp, parts = gla_layout(d, dv)
    return n_heads * dv * parts * dp


def gla_step_takes(low: torch.Tensor, w2: torch.Tensor, d: int, dv: int) -> bool:
    """Whether ``gla_scan`` forms the decays' logits of a step of single tokens itself, ``low`` [T, rank] times ``w2`` [n_heads * d, rank] transposed."""
    rank = w2.shape[1]
    if low.dtype != torch.bfloat16 or w2.dtype != torch.bfloat16 or rank % 8 or not w2.is_contiguous() or w2.data_ptr() % 16:
        return False
    if not columns_on_16_bytes(low) and (not low.is_contiguous() or low.data_ptr() % 16):
        return False
    dp, parts = gla_layout(d, dv)
    return bool(load_module("gla").fn("ifx_gla_step_takes", (I, I))(dp * parts, dv))


def gla_scan(rows: torch.Tensor, cols: Tuple[int, int, int, int], z, z_bias: Optional[torch.Tensor], tau: float,
             q_scale: float, norm_weight: torch.Tensor, eps: float, n_heads: int, d: int, dv: int, state: torch.Tensor,
             state_offset: int, q_start: torch.Tensor, q_len: torch.Tensor, slots: torch.Tensor,
             chunks: Optional[Dict[str, object]] = None) -> torch.Tensor:
    """Gated linear attention over each request's rows, with the output's norm and gate:
    alpha = sigmoid(z + z_bias) ^ (1 / tau) per key channel; per head S <- diag(alpha) S + k v^T; o = S^T q * q_scale;
    y = o / sqrt(mean(o^2) + eps) * norm_weight * silu(g).  ``rows`` [T, ld] holds q, k (n_heads * d each), v and g
    (n_heads * dv each) at the columns ``cols`` = (q, k, v, g); ``z`` float32 [T, n_heads * d], or in steps of single tokens the two factors that
    ``gla_step_takes``; ``state`` float32
    [slots, n] with a request's S (``gla_state_floats`` numbers, laid out for the kernel) at ``state_offset`` of its row.
    Decays, S, o, norm and gate are float.  Returns y [T, n_heads * dv] in the rows' type.

    ``chunks`` (from ``scan_chunks``): the requests' rows cut into chunks that run side by side, first from a zero state,
    then from the state the chunks before leave (the recurrence is linear in S); the same function up to the rounding of
    float sums taken in another order."""
    _check(rows, "rows", (None, None))
    T, ld = rows.shape
    HD, HV = n_heads * d, n_heads * dv
    q_col, k_col, v_col, g_col = (int(c) for c in cols)
    for c, w, nm in ((q_col, HD, "q"), (k_col, HD, "k"), (v_col, HV, "v"), (g_col, HV, "g")):
        if c < 0 or c + w > ld:
            raise KernelError(f"gla_scan: the {nm} columns {c}..{c + w} lie outside rows of {ld}")
    low_args = (None, 0, None, 0)
    if isinstance(z, tuple):
        low, w2 = z
        if low.shape[0] != T or w2.shape != (HD, low.shape[1]) or rows.dtype != torch.bfloat16 or T > q_start.shape[0] or chunks is not None \
                or not gla_step_takes(low, w2, d, dv):
            raise KernelError(f"gla_scan: the product of {tuple(low.shape)} and {tuple(w2.shape)} is not formed for {T} rows of {q_start.shape[0]} requests")
        low_args, z = (low, low.stride(0), w2, low.shape[1]), None
    else:
        _check(z, "z", (T, HD), torch.float32)
    if z_bias is not None:
        _check(z_bias, "z_bias", (HD,), torch.float32)
    _check(norm_weight, "norm_weight", (dv,))
    _check(state, "state", (None, None), torch.float32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    dp, parts = gla_layout(d, dv)
    if state_offset + n_heads * dv * parts * dp > state.shape[1]:
        raise KernelError("gla_scan: the state rows are too short")
    out = empty((T, HV), rows.dtype, rows)
    base, size = rows.data_ptr(), rows.element_size()
    n_chunks, lists, _keep = _chunk_lists(chunks, R, HV * parts * dp, HD, rows.device)
    _call(load_module("gla"), "ifx_gla_scan", _GLA_ARGS,
          base + q_col * size, base + k_col * size, base + v_col * size, base + g_col * size, _dt(rows), _dt(out), ld, z,
          *low_args, z_bias, 1.0 / float(tau), float(q_scale), float(eps), norm_weight, _dt(norm_weight), 0, state,
          state.shape[1], int(state_offset), q_start, q_len, slots, out, T, R, n_heads, d, dv,
          dp, parts, n_chunks, *lists, _stream())
    return out


_GLA_ARGS = (P, P, P, P, I, I, I, P, P, I, P, I, P, F, F, F, P, I, P, P, LL, LL, P, P, P, P, I, I, I, I, I, I, I, I, P, P, P, P, P, P, P)


def _chunk_lists(chunks: Optional[Dict[str, object]], R: int, state_floats: int, log_floats: int, device):
    """(number of chunks, the kernel's list arguments, what they point into) of ``gla_scan`` and ``time_mix_scan``."""
    if chunks is None:
        return 0, (0, 0, 0, 0, 0, 0), None
    n_chunks = chunks["req"].shape[0]
    for nm in ("req", "t0", "len"):
        _check(chunks[nm], f"chunks.{nm}", (n_chunks,), torch.int32)
    _check(chunks["req_chunk0"], "chunks.req_chunk0", (R + 1,), torch.int32)
    chunk_state = torch.empty((n_chunks, state_floats), dtype=torch.float32, device=device)
    chunk_loga = torch.empty((n_chunks, log_floats), dtype=torch.float32, device=device)
    return n_chunks, (chunks["req"].data_ptr(), chunks["t0"].data_ptr(), chunks["len"].data_ptr(), chunks["req_chunk0"].data_ptr(),
                      chunk_state.data_ptr(), chunk_loga.data_ptr()), (chunk_state, chunk_loga)


def _check_rows(t: torch.Tensor, name: str, T: int, width: int, dtype: Optional[torch.dtype] = None) -> int:
    """``t`` [T, width] on the GPU with contiguous rows that may lie further apart; returns their distance."""
    if not (isinstance(t, torch.Tensor) and t.is_cuda and tuple(t.shape) == (T, width) and (dtype is None or t.dtype == dtype)
            and (width == 1 or t.stride(1) == 1) and (T <= 1 or t.stride(0) >= width)):
        raise KernelError(f"{name}: needs [{T}, {width}] rows on the GPU" + (f" of {dtype}" if dtype is not None else ""))
    return t.stride(0) if T > 1 else max(t.stride(0), width)


def shifted_mixes(h: torch.Tensor, mu: torch.Tensor, state: torch.Tensor, state_offset: int, row_req: torch.Tensor, q_start: torch.Tensor,
                  q_len: torch.Tensor, slots: torch.Tensor) -> torch.Tensor:
    """[S, T, H] in h's type: h + (h' - h) mu[s] with h' the request's row before, ``mu`` float32 [S, H].  A request's last row lives
    in the H floats from ``state_offset`` of its row of ``state`` [slots, n] (float32, zero for a request that starts): it is
    read as the row before this step's first and replaced by this step's last."""
    _check(h, "h", (None, None))
    T, H = h.shape
    _check(mu, "mu", (None, H), torch.float32)
    _check(state, "state", (None, None), torch.float32)
    _check(row_req, "row_req", (T,), torch.int32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    out = empty((mu.shape[0], T, H), h.dtype, h)
    _call(load_module("time_mix"), "ifx_shifted_mixes", (P, I, P, P, LL, LL, P, P, P, P, P, I, I, I, P),
          h, _dt(h), mu, state, state.shape[1], int(state_offset), row_req, q_start,
          q_len, slots, out, T, H, mu.shape[0], _stream())
    return out


def lowrank_tanh(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """tanh(a) W in float: ``a`` float32 [T, r] (rows may lie further apart), ``w`` [r, C]; float32 [T, C]."""
    _check(w, "w", (None, None))
    r, C = w.shape
    T = a.shape[0]
    lda = _check_rows(a, "a", T, r, torch.float32)
    z = empty((T, C), torch.float32, w)
    _call(load_module("time_mix"), "ifx_lowrank_tanh", (P, I, P, I, P, I, I, I, P), a, lda, w, _dt(w), z, T, r, C,
          _stream())
    return z


def time_mix_scan(r: torch.Tensor, k: torch.Tensor, v: torch.Tensor, g: torch.Tensor, z: torch.Tensor, w0: torch.Tensor, u: torch.Tensor,
                  norm_weight: torch.Tensor, eps: float, n_heads: int, d: int, state: torch.Tensor, state_offset: int, q_start: torch.Tensor,
                  q_len: torch.Tensor, slots: torch.Tensor, out_dtype: torch.dtype, chunks: Optional[Dict[str, object]] = None) -> torch.Tensor:
    """Time mixing's recurrence over each request's rows, with the output's norm and gate: w = exp(-exp(z + w0)) per key channel;
    o = (S + diag(u) k v^T)^T r; S <- diag(w) S + k v^T; y = o / sqrt(mean(o^2) + eps) * norm_weight * silu(g).  ``r``, ``k``,
    ``v``, ``g`` [T, n_heads * d] (one element type; rows equally far apart), ``z`` float32 [T, n_heads * d], ``w0`` float32
    [n_heads * d], ``u`` float32 [n_heads, d], ``norm_weight`` float32 [n_heads * d]; ``state`` as for ``gla_scan`` (values as
    wide as keys), and ``chunks`` too.  Everything between is float.  Returns y [T, n_heads * d] in ``out_dtype``."""
    T, HD = r.shape[0], n_heads * d
    lds = [_check_rows(t, nm, T, HD, r.dtype) for t, nm in ((r, "r"), (k, "k"), (v, "v"), (g, "g"))]
    if len(set(lds)) != 1:
        raise KernelError(f"time_mix_scan: rows {lds} elements apart (they must agree)")
    _check(z, "z", (T, HD), torch.float32)
    for t, nm, shape in ((w0, "w0", (HD,)), (u, "u", (n_heads, d)), (norm_weight, "norm_weight", (HD,))):
        _check(t, nm, shape, torch.float32)
    _check(state, "state", (None, None), torch.float32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    dp, parts = gla_layout(d, d)
    if state_offset + HD * parts * dp > state.shape[1]:
        raise KernelError("time_mix_scan: the state rows are too short")
    out = empty((T, HD), out_dtype, r)
    n_chunks, lists, _keep = _chunk_lists(chunks, R, HD * parts * dp, HD, r.device)
    _call(load_module("gla", TIME_MIX), "ifx_gla_scan", _GLA_ARGS,
          r, k, v, g, _dt(r), _DT[out_dtype], lds[0], z, None, 0, None, 0, w0, 1.0, 1.0,
          float(eps), norm_weight, _dt(norm_weight), u, state, state.shape[1], int(state_offset),
          q_start, q_len, slots, out, T, R, n_heads, d, d, dp, parts, n_chunks, *lists, _stream())
    return out


# ----------------------------------------------------------------------------------------
MEMORY_THREAD_CHANNELS = (4, 8, 16, 32)     # key channels of a column of S a thread may hold
MEMORY_MAX_PADDED_DIM, MEMORY_THREADS = 512, 256
# ... at most this many in steps of single tokens whose heads are too large or too small for the kernel that takes a head whole (64 rows at 4 heads of 256 x 256: 69.0 us
MEMORY_DECODE_MAX_CHANNELS = 8              # with 4, 47.4 with 8, 48.1 with 16)


def matrix_memory_layout(d: int, dv: int, single_tokens: bool = False) -> Tuple[int, int, int]:
    """(channels a thread, threads a column, columns a workgroup) of the matrix memory's walk for heads of ``d`` key channels
    and ``dv`` values (dv + 1 columns: the last is the normaliser's), the columns dealt evenly to as many workgroups as it takes.
    The state's layout (columns of d padded to a power of two) does not depend on the choice: a walk over many tokens is
    shortest with few channels a thread, steps of single tokens want few workgroups (``single_tokens``)."""
    dpad = 4
    while dpad < d:
        dpad *= 2
    if dpad > MEMORY_MAX_PADDED_DIM:
        raise KernelError(f"matrix memory: heads of {d} key channels (at most {MEMORY_MAX_PADDED_DIM})")
    found = [(ch, dpad // ch) for ch in MEMORY_THREAD_CHANNELS if ch <= dpad and dpad // ch <= 64]
    ch, ks = found[0]
    if single_tokens:
        ch, ks = next((f for f in reversed(found) if f[0] <= MEMORY_DECODE_MAX_CHANNELS), found[0])
    most = max(1, MEMORY_THREADS // ks)
    groups = -(-(dv + 1) // most)
    return ch, ks, -(-(dv + 1) // groups)


def _memory_max_floats(n_heads: int) -> int:
    return -(-n_heads // 4) * 4         # the running maxima come first in a state row


MEMORY_CHUNK = 64                   # rows of a chunk where long portions are cut into chunks that run side by side


def matrix_memory_takes_chunks(dtype: torch.dtype, d: int, dv: int) -> bool:
    return dtype == torch.bfloat16 and d % 8 == 0 and dv % 8 == 0


def matrix_memory_state_floats(n_heads: int, d: int, dv: int) -> int:
    ch, ks, _ = matrix_memory_layout(d, dv)
    return _memory_max_floats(n_heads) + n_heads * (dv + 1) * ch * ks


def matrix_memory(rows: torch.Tensor, cols: Tuple[int, int, int, int], gates: torch.Tensor, gate_cols: Tuple[int, int], i_bias: torch.Tensor,
                  f_bias: torch.Tensor, cap: float, norm_weight: torch.Tensor, eps: float, n_heads: int, d: int, dv: int, state: torch.Tensor,
                  q_start: torch.Tensor, q_len: torch.Tensor, slots: torch.Tensor, row_req: torch.Tensor, out_dtype: torch.dtype,
                  single_tokens: bool = False, chunks: Optional[Dict[str, object]] = None) -> torch.Tensor:
    """Matrix memory with exponential gates over each request's rows, with the output's norm and gate (see
    csrc/matrix_memory.hip).  ``rows`` [T, ld] holds q, k (n_heads * d each), v and the output gate (n_heads * dv each) at the
    columns ``cols``; ``gates`` float32 [T, ldg] the input and forget gates' numbers (n_heads each) at ``gate_cols``; biases
    float32 [n_heads], ``norm_weight`` float32 [n_heads * dv].  ``state`` float32 [slots, ``matrix_memory_state_floats``], zero
    for a request that starts.  ``single_tokens``: every request brings one row.  Returns [T, n_heads * dv] in ``out_dtype``.

    ``chunks`` (from ``scan_chunks`` with MEMORY_CHUNK rows; bfloat16 rows, see ``matrix_memory_takes_chunks``): the requests'
    rows in chunks that run side by side on the matrix cores; the same function up to the rounding of float sums taken in
    another order."""
    _check(rows, "rows", (None, None))
    T, ld = rows.shape
    _check(gates, "gates", (T, None), torch.float32)
    ldg = gates.shape[1]
    HD, HV = n_heads * d, n_heads * dv
    q_col, k_col, v_col, g_col = (int(c) for c in cols)
    for c, w, nm in ((q_col, HD, "q"), (k_col, HD, "k"), (v_col, HV, "v"), (g_col, HV, "gate")):
        if c < 0 or c + w > ld:
            raise KernelError(f"matrix_memory: the {nm} columns {c}..{c + w} lie outside rows of {ld}")
    i_col, f_col = (int(c) for c in gate_cols)
    if min(i_col, f_col) < 0 or max(i_col, f_col) + n_heads > ldg:
        raise KernelError(f"matrix_memory: the gates' columns {i_col}, {f_col} lie outside rows of {ldg}")
    for t, nm, shape in ((i_bias, "i_bias", (n_heads,)), (f_bias, "f_bias", (n_heads,)), (norm_weight, "norm_weight", (HV,))):
        _check(t, nm, shape, torch.float32)
    _check(state, "state", (None, None), torch.float32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    _check(row_req, "row_req", (T,), torch.int32)
    ch, ks, wg_cols = matrix_memory_layout(d, dv, single_tokens)
    s_off = _memory_max_floats(n_heads)
    if s_off + n_heads * (dv + 1) * ch * ks > state.shape[1]:
        raise KernelError("matrix_memory: the state rows are too short")
    out = empty((T, HV), out_dtype, rows)
    scratch = empty((T * n_heads * (dv + 2) + R * n_heads,), torch.float32, rows)
    o_raw = scratch.data_ptr()
    nq = o_raw + 4 * T * n_heads * dv
    floor = nq + 4 * T * n_heads
    m_end = floor + 4 * T * n_heads
    n_chunks, lists = 0, (0,) * 7
    if chunks is not None:
        if not matrix_memory_takes_chunks(rows.dtype, d, dv) or chunks["rows"] != MEMORY_CHUNK:
            raise KernelError(f"matrix_memory: chunks of {chunks['rows']} rows of {rows.dtype} with heads of {d} x {dv} (chunks of "
                              f"{MEMORY_CHUNK} rows of bfloat16, heads of multiples of 8)")
        n_chunks = chunks["req"].shape[0]
        for nm in ("req", "t0", "len"):
            _check(chunks[nm], f"chunks.{nm}", (n_chunks,), torch.int32)
        _check(chunks["req_chunk0"], "chunks.req_chunk0", (R + 1,), torch.int32)
        gates_scratch = empty((3 * n_heads * T + 2 * n_heads * n_chunks,), torch.float32, rows)
        chunk_state = empty((n_chunks, n_heads * (dv + 1) * ch * ks), torch.float32, rows)
        lists = (chunks["req"].data_ptr(), chunks["t0"].data_ptr(), chunks["len"].data_ptr(), chunks["req_chunk0"].data_ptr(),
                 gates_scratch.data_ptr(), gates_scratch.data_ptr() + 12 * n_heads * T, chunk_state.data_ptr())
    _call(load_module("matrix_memory"), "ifx_matrix_memory",
          (P, I, I, I, I, I, I, P, I, I, I, P, P, F, F, P, F, P, LL, I, P, P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, I, I, I, P, P, P, P, P, P, P, P),
          rows, _dt(rows), ld, q_col, k_col, v_col, g_col, gates, ldg, i_col, f_col, i_bias,
          f_bias, float(cap), float(d) ** -0.5, norm_weight, float(eps), state, state.shape[1], s_off,
          q_start, q_len, slots, row_req, o_raw, nq, floor, m_end, out, _DT[out_dtype],
          T, R, n_heads, d, dv, ch, ks, wg_cols, n_chunks, *lists, _stream())
    return out


# ----------------------------------------------------------------------------------------
RETENTION_THREAD_CHANNELS = (4, 8, 16)      # key channels of a column of S a thread of the walk may hold
RETENTION_MAX_PADDED_DIM, RETENTION_MAX_VALUES = 512, 4096
RETENTION_CHUNK = 64                # rows of a chunk where long portions are cut into chunks that run side by side


def retention_layout(d: int, dv: int) -> Tuple[int, int, int]:
    """(channels a thread, threads a column, columns a workgroup) of the walk for heads of ``d`` key channels and ``dv`` values,
    the columns dealt evenly to as many workgroups as it takes.  A column of S is padded to the power of two from 4 on that
    holds d."""
    dpad = 4
    while dpad < d:
        dpad *= 2
    if dpad > RETENTION_MAX_PADDED_DIM or dv > RETENTION_MAX_VALUES:
        raise KernelError(f"retention: heads of {d} key channels and {dv} values (at most {RETENTION_MAX_PADDED_DIM} and {RETENTION_MAX_VALUES})")
    ch, ks = next((ch, dpad // ch) for ch in RETENTION_THREAD_CHANNELS if dpad // ch <= 64)
    most = max(1, 256 // ks)
    groups = -(-dv // most)
    return ch, ks, -(-dv // groups)


def retention_step_columns(n_rows: int, n_heads: int, d: int, dv: int) -> int:
    """Columns of a head that a workgroup takes in a step of single tokens: all of them (one launch finishes the head), unless the
    heads are large and so few that a workgroup each would leave most of the chip idle."""
    ch, ks, _ = retention_layout(d, dv)
    heads, columns = max(n_rows * n_heads, 1), dv
    while columns * ch * ks > 16384 and heads * -(-dv // columns) < 128:
        columns = -(-columns // 2)
    return columns


def retention_state_floats(n_heads: int, d: int, dv: int) -> int:
    ch, ks, _ = retention_layout(d, dv)
    return n_heads * dv * ch * ks


def retention_takes_chunks(dtype: torch.dtype, d: int, dv: int) -> bool:
    return dtype == torch.bfloat16 and d % 8 == 0 and dv % 8 == 0


def retention(rows: torch.Tensor, cols: Tuple[int, int, int, int], cos: torch.Tensor, sin: torch.Tensor, rot_dims: int, decay: torch.Tensor,
              log2_decay: torch.Tensor, eps: float, n_heads: int, d: int, dv: int, state: torch.Tensor, q_start: torch.Tensor,
              q_len: torch.Tensor, slots: torch.Tensor, out_dtype: torch.dtype, single_tokens: bool = False,
              chunks: Optional[Dict[str, object]] = None) -> torch.Tensor:
    """Retention over each request's rows, with the turn of q and k before it and the heads' norm and gate behind it (see
    csrc/retention.hip).  ``rows`` [T, ld] holds q, k (n_heads * d each), v and the output gate (n_heads * dv each) at the columns
    ``cols``; the first ``rot_dims`` channels of every q and k head turn by the table ``cos`` / ``sin`` float32 [T, rot_dims / 2];
    ``decay`` and ``log2_decay`` float32 [n_heads].  ``state`` float32 [slots, ``retention_state_floats``], zero for a request that
    starts.  ``single_tokens``: every request brings one row.  Returns [T, n_heads * dv] in ``out_dtype``.

    ``chunks`` (from ``scan_chunks`` with RETENTION_CHUNK rows; bfloat16 rows, see ``retention_takes_chunks``): the requests' rows
    in chunks that run side by side on the matrix cores; the same function up to the rounding of float sums taken in another
    order."""
    _check(rows, "rows", (None, None))
    T, ld = rows.shape
    HD, HV = n_heads * d, n_heads * dv
    q_col, k_col, v_col, g_col = (int(c) for c in cols)
    for c, w, nm in ((q_col, HD, "q"), (k_col, HD, "k"), (v_col, HV, "v"), (g_col, HV, "gate")):
        if c < 0 or c + w > ld:
            raise KernelError(f"retention: the {nm} columns {c}..{c + w} lie outside rows of {ld}")
    if rot_dims % 2 or not 0 <= rot_dims <= d:
        raise KernelError(f"retention: {rot_dims} of {d} channels turn")
    for t, nm in ((cos, "cos"), (sin, "sin")):
        if rot_dims:
            _check(t, nm, (T, rot_dims // 2), torch.float32)
    _check(decay, "decay", (n_heads,), torch.float32)
    _check(log2_decay, "log2_decay", (n_heads,), torch.float32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (slots, "slots")):
        _check(t, nm, (R,), torch.int32)
    ch, ks, wg_cols = retention_layout(d, dv)
    _check(state, "state", (None, n_heads * dv * ch * ks), torch.float32)
    if single_tokens and T != R:
        raise KernelError(f"retention: {T} rows of {R} requests are no step of single tokens")
    out = empty((T, HV), out_dtype, rows)
    n_chunks, lists, o_raw = 0, (0,) * 5, None
    if chunks is not None:
        if not retention_takes_chunks(rows.dtype, d, dv) or chunks["rows"] != RETENTION_CHUNK:
            raise KernelError(f"retention: chunks of {chunks['rows']} rows of {rows.dtype} with heads of {d} x {dv} (chunks of "
                              f"{RETENTION_CHUNK} rows of bfloat16, heads of multiples of 8)")
        n_chunks = chunks["req"].shape[0]
        for nm in ("t0", "len"):
            _check(chunks[nm], f"chunks.{nm}", (n_chunks,), torch.int32)
        _check(chunks["req_chunk0"], "chunks.req_chunk0", (R + 1,), torch.int32)
        turned = empty((4, T * HD), torch.bfloat16, rows)
        chunk_state = empty((n_chunks, n_heads * dv * ch * ks), torch.float32, rows)
        lists = (chunks["t0"].data_ptr(), chunks["len"].data_ptr(), chunks["req_chunk0"].data_ptr(), turned.data_ptr(), chunk_state.data_ptr())
    if single_tokens and chunks is None:
        wg_cols = retention_step_columns(T, n_heads, d, dv)
    if (chunks is None and (not single_tokens or wg_cols < dv)) or (chunks is not None and dv > 128):
        o_raw = empty((T, HV), torch.float32, rows)
    _call(load_module("retention"), "ifx_retention",
          (P, I, I, I, I, I, I, P, P, I, P, P, F, F, P, LL, P, P, P, P, P, I, I, I, I, I, I, I, I, I, I, I, P, P, P, P, P, P),
          rows, _dt(rows), ld, q_col, k_col, v_col, g_col, cos if rot_dims else None, sin if rot_dims else None, rot_dims // 2,
          decay, log2_decay, float(d) ** -0.5, float(eps), state, state.shape[1], q_start,
          q_len, slots, o_raw, out, _DT[out_dtype], T, R, n_heads, d, dv, ch, ks, wg_cols,
          1 if single_tokens else 0, n_chunks, *lists, _stream())
    return out


HYPER_MAX_STREAMS = 8


def hyper_step(src: torch.Tensor, n_streams: int, y=None, mix: Optional[torch.Tensor] = None, out_weights: Optional[torch.Tensor] = None,
               in_weights: Optional[torch.Tensor] = None, norm_weight: Optional[torch.Tensor] = None, eps: float = 0.0,
               out_dtype: Optional[torch.dtype] = None, y_scale: float = 1.0):
    """One step of hyper-connections on the streams of a step's rows, in float.

    ``src`` float32: the streams [T, S, H], or one stream [T, H] that all S start as.  With ``y`` [T, H] (a tensor of any
    activation type or ``SliceSums``) the streams become x_t <- sum_s mix[s, t] x_s + out_weights[t] * y * y_scale, in
    place (copies of a single stream are written to a new tensor).  With ``in_weights`` the sub-block that follows reads
    u = sum_t in_weights[t] x_t of the new streams: returned normalised, u / sqrt(mean(u^2) + eps) * norm_weight in
    ``out_dtype``, or as it is in float32 without ``norm_weight``.  Returns (streams, rows or None)."""
    S = int(n_streams)
    single = src.dim() == 2
    if single:
        _check(src, "src", (None, None), torch.float32)
        T, H = src.shape
    else:
        _check(src, "src", (None, S, None), torch.float32)
        T, _, H = src.shape
    if not 0 < S <= HYPER_MAX_STREAMS:
        raise KernelError(f"hyper_step: {S} streams (1 to {HYPER_MAX_STREAMS})")
    for t, nm, shape in ((mix, "mix", (S, S)), (out_weights, "out_weights", (S,)), (in_weights, "in_weights", (S,))):
        if t is not None:
            _check(t, nm, shape, torch.float32)
    n_slices, stride, y_ptr, y_dt = 1, 0, 0, 0
    if y is not None:
        if mix is None or out_weights is None:
            raise KernelError("hyper_step: an update needs the mixing matrix and the output weights")
        if isinstance(y, SliceSums):
            _check(y.parts, "y", (None, T, H), torch.float32)
            n_slices, stride, y_ptr, y_dt = y.parts.shape[0], T * H, y.parts.data_ptr(), DT_F32
        else:
            _check(y, "y", (T, H))
            y_ptr, y_dt = y.data_ptr(), _dt(y)
    dst = empty((T, S, H), torch.float32, src) if single else src
    rows = None
    if in_weights is not None:
        if norm_weight is not None:
            _check(norm_weight, "norm_weight", (H,))
            rows = torch.empty((T, H), dtype=out_dtype or torch.float32, device=src.device)
        else:
            rows = empty((T, H), torch.float32, src)
    _call(load_module("hyper"), "ifx_hyper_step", (P, I, P, P, I, I, LL, F, P, P, P, P, I, F, P, I, I, I, I, P),
          src, 1 if single else 0, dst, y_ptr, y_dt, n_slices, stride, float(y_scale), mix, out_weights,
          in_weights, norm_weight, _dt(norm_weight) if norm_weight is not None else 0, float(eps), rows,
          _DT[rows.dtype] if rows is not None else 0, T, S, H, _stream())
    return dst, rows


def linear_act(x, weight, act: int) -> torch.Tensor:
    """act(x W^T) for a feed-forward without a gate (``act``: ACT_SILU, ACT_GELU_TANH or ACT_RELU_SQUARED, formed in float on the product's
    output; in steps of few rows the square of relu and gelu are the product's epilogue: 16 rows of 8,448 x 2,048 12 us and a launch of 5 less,
    in those of many rows any of them: ``many_tiles_take``);
    ``x`` as for ``linear``."""
    if act in _PLAIN_EPILOGUE and isinstance(weight, LinearWeight) and weight.rows.dtype == torch.bfloat16 and x.dtype == torch.bfloat16 \
            and weight.order is None and _small_m_kernel(x.shape[0], *weight.rows.shape, weight.tiled is not None) == "skinny" \
            and (not isinstance(x, ScaledRows) or takes_scaled_rows(x.shape[0], weight)):
        if ring_takes_few(x, weight):
            return ring_gemm(x, weight, plain_act=act)
        return skinny_gemm(x, weight.rows, tiled=weight.tiled, tile_rows=weight.tile_rows, plain_act=act)
    rows = weight.rows if isinstance(weight, LinearWeight) else weight
    if not isinstance(x, ScaledRows) and rows.dtype == torch.bfloat16 and x.dtype == torch.bfloat16 and rows.dim() == 2 and x.dim() == 2 \
            and x.shape[1] == rows.shape[1] and act in PLAIN_ACTS and many_tiles_take(x.shape[0], *rows.shape, gated=False):
        whole = x.contiguous() if columns_on_16_bytes(x) else x          # (as for ``linear``)
        if whole.is_contiguous() and whole.data_ptr() % 16 == 0 and rows.is_contiguous() and rows.data_ptr() % 16 == 0:
            return act_tiles(whole, rows, act)
    return activation(linear(x, weight, keep_slices=True), act)


def activation(x, act: int) -> torch.Tensor:
    """act(x) element by element in float: ACT_SILU, ACT_GELU_TANH or ACT_RELU_SQUARED (a feed-forward without a gate).  ``x`` may be
    ``SliceSums``: the partial sums are added in slice order first, and the result has the type they stand for."""
    if isinstance(x, SliceSums):
        parts = x.parts
        _check(parts, "x", (None, None, None), torch.float32)
        n = parts.shape[1] * parts.shape[2]
        if n % 4:
            return activation(x.sum(x.dtype), act)
        out = torch.empty(parts.shape[1:], dtype=x.dtype, device=parts.device)
        _call(load_module("rowwise"), "ifx_activation_slices", (P, I, LL, P, I, LL, I, P), parts, parts.shape[0], n,
              out, _DT[x.dtype], n, int(act), _stream())
        return out
    _check(x, "x")
    out = torch.empty_like(x)
    _call(load_module("rowwise"), "ifx_activation", (P, P, I, LL, I, P), x, out, _dt(x), x.numel(), int(act), _stream())
    return out


def sigmoid_gate(x: torch.Tensor, rows, g_col: int) -> torch.Tensor:
    """x [T, C] times sigmoid of the columns ``g_col`` .. ``g_col`` + C - 1 of ``rows`` [T, ld] (x's type, or ``SliceSums``),
    element by element, the sigmoid in float."""
    _check(x, "x", (None, None))
    T, C = x.shape
    n_slices = stride = 0
    if isinstance(rows, SliceSums):
        _check(rows.parts, "rows", (None, T, None), torch.float32)
        n_slices, ld, stride, ptr = rows.parts.shape[0], rows.parts.shape[2], T * rows.parts.shape[2], rows.parts.data_ptr()
    else:
        _check(rows, "rows", (T, None), x.dtype)
        ld, ptr = rows.shape[1], rows.data_ptr()
    if g_col < 0 or g_col + C > ld:
        raise KernelError(f"sigmoid_gate: columns {g_col}..{g_col + C} lie outside rows of {ld}")
    out = torch.empty_like(x)
    _call(load_module("rowwise"), "ifx_sigmoid_gate", (P, P, I, I, I, LL, P, I, I, I, P),
          x, ptr, ld, int(g_col), n_slices, stride, out, _dt(x), T, C, _stream())
    return out


def gated_add(base, extra, h: torch.Tensor, gate_weight: Optional[torch.Tensor]) -> torch.Tensor:
    """base + sigmoid(h . gate_weight) * extra row by row: ``base`` and ``extra`` [T, N] (h's type, or ``SliceSums``, which are
    added in slice order), ``h`` [T, K], ``gate_weight`` [K] (one number per row, formed in float; None: the gate is 1, and
    ``h`` only says the type and the number of rows).  Returns [T, N] in h's type."""
    _check(h, "h", (None, None))
    T, K = h.shape
    if gate_weight is not None:
        _check(gate_weight, "gate_weight", (K,), h.dtype)

    def operand(v, nm):
        if isinstance(v, SliceSums):
            _check(v.parts, nm, (None, T, None), torch.float32)
            return v.parts.data_ptr(), 1, v.parts.shape[0], T * v.parts.shape[2], v.parts.shape[2]
        _check(v, nm, (T, None), h.dtype)
        return v.data_ptr(), 1 if v.dtype == torch.float32 else 0, 1, 0, v.shape[1]

    bp, bf, bn, bs, N = operand(base, "base")
    ep, ef, en, es, N2 = operand(extra, "extra")
    if N != N2:
        raise KernelError(f"gated_add: base is {N} wide, extra {N2}")
    out = empty((T, N), h.dtype, h)
    _call(load_module("rowwise"), "ifx_gated_add", (P, I, I, LL, P, I, I, LL, P, P, I, P, I, I, I, P),
          bp, bf, bn, bs, ep, ef, en, es, h, gate_weight, K, out, _dt(h), T, N, _stream())
    return out


def scale_softcap(logits: torch.Tensor, scale: float = 1.0, cap: float = 0.0) -> torch.Tensor:
    """In place on float32 ``logits``: x <- x * scale, then (cap > 0) x <- cap * tanh(x / cap)."""
    _check(logits, "logits", None, torch.float32)
    _call(load_module("rowwise"), "ifx_scale_softcap", (P, LL, F, F, P), logits, logits.numel(), float(scale), float(cap or 0.0), _stream())
    return logits


WIDE_MAX_K_DIM, WIDE_MAX_V_DIM = 1024, 512
WIDE_DIMS_PREBUILT = ((576, 512),)      # compiled ahead by build_all(); any other pair of widths when a model first needs it


def wide_attention_supported(dtype: torch.dtype, n_kv_heads: int, k_dim: int, v_dim: int, page_size: int) -> bool:
    """Whether ``attention_wide`` takes this cache: bfloat16, one kv head that all query heads share, keys of a multiple
    of 8 and values of a multiple of 16 elements, pages of a power of two from 16."""
    return (dtype == torch.bfloat16 and n_kv_heads == 1 and k_dim % 8 == 0 and 0 < k_dim <= WIDE_MAX_K_DIM and v_dim % 16 == 0
            and 0 < v_dim <= WIDE_MAX_V_DIM and page_size >= 16 and page_size & (page_size - 1) == 0)


def wide_launch_shape(n_rows: int, n_heads: int, max_kv: int):
    """(keys per split, splits) of a launch of ``attention_wide``: one wave per (row, 16 heads, split), splits as long as
    still give the chip about 2,048 waves, and no shorter than 64 keys."""
    groups = -(-n_heads // 16)
    splits = max(1, min(2048 // max(n_rows * groups, 1), -(-max_kv // 64)))
    chunk = max(64, -(-(-(-max_kv // splits)) // 32) * 32)
    return chunk, max(1, -(-max_kv // chunk))


def attention_wide(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, row_req: torch.Tensor, positions: torch.Tensor,
                   block_table: torch.Tensor, window: Optional[int], scale: float, chunk: int, max_splits: int,
                   sinks: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal (optionally windowed) attention of q [T, nH, d] over one shared kv head with keys of d and values of dv
    elements (K [pages, 1, page, d], V [pages, 1, dv, page]) on the matrix cores, for widths the other matrix-core kernels
    do not take; returns [T, nH * dv].  Every row's keys are cut into splits of ``chunk`` (``max_splits`` * chunk must
    reach past the largest position) and merged by a second launch.  ``sinks`` float32 [nH]: a score per head that joins
    its softmax's denominator."""
    _check(q, "q", (None, None, None), torch.bfloat16)
    T, nH, d = q.shape
    if sinks is not None:
        _check(sinks, "sinks", (nH,), torch.float32)
    _check(k_cache, "k_cache", (None, 1, None, d), torch.bfloat16)
    n_pages, _, page_size, _ = k_cache.shape
    _check(v_cache, "v_cache", (n_pages, 1, None, page_size), torch.bfloat16)
    dv = v_cache.shape[2]
    if not wide_attention_supported(q.dtype, 1, d, dv, page_size):
        raise KernelError(f"attention_wide: keys of {d} (a multiple of 8 up to {WIDE_MAX_K_DIM}), values of {dv} (of 16 up to "
                          f"{WIDE_MAX_V_DIM}), pages of {page_size} (a power of two from 16)")
    _check(row_req, "row_req", (T,), torch.int32)
    _check(positions, "positions", (T,), torch.int32)
    _check(block_table, "block_table", (None, None), torch.int32)
    out = empty((T, nH * dv), torch.bfloat16, q)
    part_o = empty((T, nH, max_splits, dv), torch.float32, q)
    part_ml = empty((T, nH, max_splits, 2), torch.float32, q)
    _call(load_module("attn_wide", (("K_DIM", d), ("V_DIM", dv))), "ifx_attn_wide",
          (P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, I, I, F, P, P, P, P),
          q, k_cache, v_cache, out, 0, row_req, positions,
          block_table, block_table.shape[1], T, nH, d, dv, page_size, int(window or 0), int(chunk), int(max_splits),
          float(scale), part_o, part_ml, sinks, _stream())
    return out


def mfma_attention_supported(dtype: torch.dtype, head_dim: int, page_size: int) -> bool:
    return (dtype == torch.bfloat16 and head_dim % 16 == 0 and head_dim <= MFMA_MAX_HEAD_DIM
            and page_size >= 16 and page_size & (page_size - 1) == 0)


def _attn_common(q, k_cache, v_cache, qt=1, direct=True):
    _check(q, "q", (None, None, None), torch.bfloat16)
    T, nH, d = q.shape
    _check(k_cache, "k_cache", (None, None, None, d), torch.bfloat16)
    n_pages, nKV, page_size, _ = k_cache.shape
    _check(v_cache, "v_cache", (n_pages, nKV, d, page_size), torch.bfloat16)
    if not mfma_attention_supported(q.dtype, d, page_size):
        raise KernelError(f"matrix-core attention needs bfloat16, head_dim a multiple of 16 up to {MFMA_MAX_HEAD_DIM} and "
                          f"page_size a power of two from 16; got head_dim {d}, page_size {page_size}")
    name, variant, _, _ = _tile_module(d, qt, direct)
    return T, nH, d, nKV, page_size, load_module(name, variant)


def _attn_extras(T, nH, keep_first, sink, gate, sinks=None, block=None):
    """The six optional arguments of the matrix-core attention kernels: kept first keys, whether there is a sink, its
    score, the gate's pointer, the pointer to a sink score per head, the size of the blocks a row sees its own of."""
    if gate is not None:
        _check(gate, "gate", (T, nH), torch.float32)
    if sinks is not None:
        _check(sinks, "sinks", (nH,), torch.float32)
    return int(keep_first or 0), 0 if sink is None else 1, float(sink or 0.0), gate, sinks, int(block or 0)


ROW_MAX_WAVES = 8


def row_waves_fit(n_heads: int, n_kv_heads: int, head_dim: int, waves: int) -> int:
    """The most waves per workgroup, up to ``waves``, whose results fit the row kernel's 64 KB of LDS."""
    nc = min(16, n_heads // n_kv_heads)
    while waves > 1 and waves * nc * (head_dim + 6) * 4 > 65536:
        waves //= 2
    return waves


def attention_rows(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, out: torch.Tensor,
                   rows: Optional[torch.Tensor], n_rows: int, row_req: torch.Tensor, positions: torch.Tensor,
                   block_table: torch.Tensor, window: Optional[int], scale: float, chunk: int, max_splits: int,
                   waves: int = 0, req_is_row: bool = False, keep_first: int = 0, sink: Optional[float] = None,
                   gate: Optional[torch.Tensor] = None, sinks: Optional[torch.Tensor] = None, block: Optional[int] = None) -> Optional["SplitRows"]:
    """Attention of single rows (``rows`` int32, or None for rows 0..n_rows-1) into ``out`` [T, nH*d].  ``keep_first``,
    ``sink``, ``gate``: as for ``attention_plain``.  Without ``out`` (every row, in splits, no ``sink`` and no ``gate``) the splits are left
    to the reader and returned.

    ``waves`` 0: split s of a row covers key positions [s*chunk, (s+1)*chunk), one wave each, and a second launch
    merges a row's splits; ``max_splits`` * chunk must reach past the largest position among the rows.
    ``waves`` 1-8: one workgroup of that many waves per (row, kv head) shares the row's keys evenly and writes the
    output itself (``chunk`` and ``max_splits`` are not used): for launches with pairs enough to fill the chip.
    ``req_is_row``: the caller vouches that ``row_req`` is 0, 1, 2, ... (every request brings one row), which lets
    a wave ask for its block-table entries before it knows anything else."""
    T, nH, d, nKV, page_size, mod = _attn_common(q, k_cache, v_cache)
    if out is not None:
        _check(out, "out", (T, nH * d), torch.bfloat16)
    elif rows is not None or waves or sink is not None or gate is not None or not 0 < max_splits <= SPLITS_READ_MAX:
        raise KernelError(f"attention_rows: {max_splits} splits are not left to the reader (1-{SPLITS_READ_MAX} of every row, no sink, no gate)")
    _check(row_req, "row_req", (T,), torch.int32)
    _check(positions, "positions", (T,), torch.int32)
    _check(block_table, "block_table", (None, None), torch.int32)
    if rows is not None:
        _check(rows, "rows", (n_rows,), torch.int32)
    elif n_rows != T:
        raise KernelError("attention_rows: without a row list every row of the batch is handled")
    if not 0 <= waves <= ROW_MAX_WAVES or row_waves_fit(nH, nKV, d, waves) != waves:
        raise KernelError(f"attention_rows: {waves} waves per workgroup (0-{ROW_MAX_WAVES}, and their results within 64 KB of LDS: "
                          f"up to {row_waves_fit(nH, nKV, d, ROW_MAX_WAVES)} at these head counts)")
    part_o = part_ml = None
    if waves == 0:
        part_o = empty((n_rows, nH, max_splits, d), torch.float32, q)
        part_ml = empty((n_rows, nH, max_splits, 2), torch.float32, q)
    if req_is_row and block_table.shape[0] < T:
        raise KernelError("attention_rows: req_is_row needs a block-table row for every row of the step")
    _call(mod, "ifx_attn_rows", (P, P, P, P, P, P, P, P, I, I, I, I, I, I, I, I, I, F, P, P, I, I, I, I, F, P, P, I, I, P),
          q, k_cache, v_cache, out, rows, row_req,
          positions, block_table, block_table.shape[1], n_rows, nH, nKV, d, page_size,
          int(window or 0), chunk, max_splits, float(scale), part_o, part_ml, waves, 1 if req_is_row else 0,
          *_attn_extras(T, nH, keep_first, sink, gate, sinks, block), 0 if out is None else 1, _stream())
    return SplitRows(part_o, part_ml, sinks) if out is None else None


def attention_tile_rows(head_dim: int, qt: int = 1) -> int:
    """Rows per tile of the tile kernel in tiling ``qt`` (see TILE_QTS; the compiled module says the same; asking it
    would compile a variant that a short step never runs)."""
    return 64 * qt


def attention_tiles(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, out: torch.Tensor,
                    tile_req: torch.Tensor, tile_q0: torch.Tensor, q_start: torch.Tensor, q_len: torch.Tensor,
                    kv_len: torch.Tensor, block_table: torch.Tensor, window: Optional[int], scale: float,
                    qt: int = 1, chunk: int = 0, max_splits: int = 1, rows: Optional[torch.Tensor] = None,
                    row_req: Optional[torch.Tensor] = None, positions: Optional[torch.Tensor] = None,
                    order: Optional[torch.Tensor] = None, keep_first: int = 0, sink: Optional[float] = None,
                    gate: Optional[torch.Tensor] = None, sinks: Optional[torch.Tensor] = None, block: Optional[int] = None, groups: int = 1,
                    beside: Optional[torch.Tensor] = None) -> None:
    """Attention of tiles of ``attention_tile_rows(d, qt)`` consecutive rows of one request each (tile t:
    request tile_req[t], rows from tile_q0[t] of that request's rows in this step) into ``out`` [T, nH*d].

    With ``max_splits`` > 1 every tile's keys are cut into splits of ``chunk`` keys (a multiple of 64;
    ``max_splits`` * chunk must reach past the largest position) that run as workgroups of their own, and
    the rows named by ``rows`` (int32: every row of every tiled request) are merged at the end; this
    needs the step's ``row_req`` and ``positions`` [T].

    ``order`` (int32 [8 * n], from ``attention.tile_order``) says which work item each workgroup of the launch
    takes; every item must appear exactly once (-1: a workgroup without work).  The result does not depend on it.

    ``groups`` 2 (``qt`` 1, one split): eight waves to a workgroup, two groups of which share its keys, for launches of fewer workgroups than
    compute units.  ``beside`` (int32, with ``groups`` 2 and the step's ``row_req`` and ``positions``, not with ``keep_first``): further rows, taken whole
    by a workgroup for each kv head in the same launch."""
    extras = bool(keep_first) or bool(block) or groups > 1      # (the kernel that loads straight into LDS has none of them)
    if groups not in (1, 2) or (groups == 2 and (qt != 1 or max_splits > 1)):
        raise KernelError(f"attention_tiles: {groups} groups of waves with tiling {qt} and {max_splits} splits (2: tiles of 64 rows, one split)")
    T, nH, d, nKV, page_size, mod = _attn_common(q, k_cache, v_cache, qt, not extras)
    _, _, entry, rows_fn = _tile_module(d, qt, not extras)
    if mod.fn(rows_fn, ())() != attention_tile_rows(d, qt):
        raise KernelError("attention_tiles: the compiled module's tile rows differ from attention_tile_rows()")
    _check(out, "out", (T, nH * d), torch.bfloat16)
    n_tiles = tile_req.shape[0]
    _check(tile_req, "tile_req", (n_tiles,), torch.int32)
    _check(tile_q0, "tile_q0", (n_tiles,), torch.int32)
    R = q_start.shape[0]
    for t, nm in ((q_start, "q_start"), (q_len, "q_len"), (kv_len, "kv_len")):
        _check(t, nm, (R,), torch.int32)
    _check(block_table, "block_table", (R, None), torch.int32)
    part_o = part_ml = None
    n_rows = n_beside = 0
    if beside is not None:
        n_beside = beside.shape[0]
        if groups != 2 or keep_first or row_req is None or positions is None or n_beside == 0:
            raise KernelError("attention_tiles: rows beside the tiles go with two groups of waves, row_req and positions, and without kept first keys")
        _check(beside, "beside", (n_beside,), torch.int32)
        _check(row_req, "row_req", (T,), torch.int32)
        _check(positions, "positions", (T,), torch.int32)
    if max_splits > 1:
        if chunk <= 0 or chunk % 64:
            raise KernelError(f"attention_tiles: splits need a chunk that is a multiple of 64, got {chunk}")
        if rows is None or row_req is None or positions is None:
            raise KernelError("attention_tiles: splits need the rows to merge, row_req and positions")
        n_rows = rows.shape[0]
        _check(rows, "rows", (n_rows,), torch.int32)
        _check(row_req, "row_req", (T,), torch.int32)
        _check(positions, "positions", (T,), torch.int32)
        part_o = empty((T, nH, max_splits, d), torch.float32, q)
        part_ml = empty((T, nH, max_splits, 2), torch.float32, q)
    per_xcd = 0
    if order is not None:
        _check(order, "order", (None,), torch.int32)
        if order.shape[0] % N_XCD:
            raise KernelError(f"attention_tiles: the order has a place for each of {N_XCD} XCDs' workgroups")
        per_xcd = order.shape[0] // N_XCD
    args = (q, k_cache, v_cache, out, tile_req, tile_q0, n_tiles, q_start, q_len, kv_len, block_table,
            block_table.shape[1], nH, nKV, d, page_size, int(window or 0), float(scale), int(chunk), int(max_splits),
            part_o, part_ml, rows, n_rows, row_req, positions, order, per_xcd, N_XCD)
    types = (P, P, P, P, P, P, I, P, P, P, P, I, I, I, I, I, I, F, I, I, P, P, P, I, P, P, P, I, I)
    if entry == "ifx_attn_tiles":
        _call(mod, entry, types + (I, I, F, P, P, I, I, P, I, P), *args, *_attn_extras(T, nH, keep_first, sink, gate, sinks, block), groups, beside, n_beside,
              _stream())
    else:
        _call(mod, entry, types + (I, F, P, P, P), *args, *_attn_extras(T, nH, 0, sink, gate, sinks)[1:5], _stream())


# ----------------------------------------------------------------------------------------
def argmax(logits: torch.Tensor) -> torch.Tensor:
    """Lowest index of the maximum of each row of float32 ``logits`` [R, V]; int32 [R]."""
    _check(logits, "logits", (None, None), torch.float32)
    R, V = logits.shape
    out = empty((R,), torch.int32, logits)
    pv = empty((R, 32), torch.float32, logits)
    pi = empty((R, 32), torch.int32, logits)
    _call(load_module("sampling"), "ifx_argmax", (P, I, I, P, P, P, P), logits, R, V, out,
          pv, pi, _stream())
    return out


def apply_penalties(logits: torch.Tensor, rows: torch.Tensor, ids: torch.Tensor, counts: torch.Tensor,
                    rep: torch.Tensor, freq: torch.Tensor, pres: torch.Tensor) -> None:
    _check(logits, "logits", (None, None), torch.float32)
    R, V = logits.shape
    n = rows.shape[0]
    for t, nm in ((rows, "rows"), (ids, "ids"), (counts, "counts")):
        _check(t, nm, (n,), torch.int32)
    for t, nm in ((rep, "rep"), (freq, "freq"), (pres, "pres")):
        _check(t, nm, (R,), torch.float32)
    _call(load_module("sampling"), "ifx_apply_penalties", (P, I, P, P, P, I, P, P, P, P),
          logits, V, rows, ids, counts, n, rep,
          freq, pres, _stream())


def add_logit_bias(logits: torch.Tensor, rows: torch.Tensor, ids: torch.Tensor, bias: torch.Tensor) -> None:
    _check(logits, "logits", (None, None), torch.float32)
    n = rows.shape[0]
    _check(rows, "rows", (n,), torch.int32)
    _check(ids, "ids", (n,), torch.int32)
    _check(bias, "bias", (n,), torch.float32)
    _call(load_module("sampling"), "ifx_add_logit_bias", (P, I, P, P, P, I, P),
          logits, logits.shape[1], rows, ids, bias, n, _stream())


def sample(logits: torch.Tensor, temperature: torch.Tensor, top_k: torch.Tensor, top_p: torch.Tensor,
           min_p: torch.Tensor, uniform: Optional[torch.Tensor] = None, draws: Optional[torch.Tensor] = None,
           any_greedy: bool = True, any_filters: bool = True) -> torch.Tensor:
    """One token per row of float32 ``logits`` [R, V]; rows with temperature <= 0 take the argmax (``any_greedy``
    False: the caller knows that there is no such row; ``any_filters`` False: that no row has top-k or top-p; both
    save launches that would find nothing to do).  The number in
    [0, 1) that a row's draw uses is either given (``uniform`` [R]) or made by the kernel from ``draws`` (int32
    [R, 4]: the row's seed and the count of its draws so far, 64 bits each, low word first), as
    ``sampling.params.philox_uniform`` makes it."""
    _check(logits, "logits", (None, None), torch.float32)
    R, V = logits.shape
    _check(temperature, "temperature", (R,), torch.float32)
    _check(top_k, "top_k", (R,), torch.int32)
    _check(top_p, "top_p", (R,), torch.float32)
    _check(min_p, "min_p", (R,), torch.float32)
    if (uniform is None) == (draws is None):
        raise KernelError("sample: either uniform numbers or seeds and counters")
    if uniform is not None:
        _check(uniform, "uniform", (R,), torch.float32)
    else:
        _check(draws, "draws", (R, 4), torch.int32)
    mod = load_module("sampling")
    weights = torch.empty_like(logits)
    out = empty((R,), torch.int32, logits)
    # large vocabularies are drawn by several workgroups a row, which hand each other their results in scratch memory
    n_scratch = mod.fn("ifx_sample_scratch_blocks", (I, I, I))(R, V, 1 if any_filters else 0)
    scratch = empty((n_scratch * 256,), torch.uint8, logits) if n_scratch else None
    _call(mod, "ifx_sample", (P, P, P, P, P, P, P, P, P, I, I, P, I, I, P),
          logits, weights, temperature, top_k, top_p,
          min_p, uniform,
          draws, out, R, V, scratch, 1 if any_greedy else 0,
          1 if any_filters else 0, _stream())
    return out


def logprobs(logits: torch.Tensor, chosen: torch.Tensor, top_n: int):
    """log-softmax of the chosen token of each row and the row's ``top_n`` (<= 20) most probable tokens:
    (lp [R], top_ids [R, top_n] int32, top_lp [R, top_n]), descending, lowest index first among equals."""
    _check(logits, "logits", (None, None), torch.float32)
    R, V = logits.shape
    _check(chosen, "chosen", (R,), torch.int32)
    lp = empty((R,), torch.float32, logits)
    top_ids = empty((R, top_n), torch.int32, logits)
    top_lp = empty((R, top_n), torch.float32, logits)
    _call(load_module("sampling"), "ifx_logprobs", (P, P, I, I, I, P, P, P, P),
          logits, chosen, R, V, top_n, lp, top_ids, top_lp, _stream())
    return lp, top_ids, top_lp


# ----------------------------------------------------------------------------------------
_SINKS: Dict[int, torch.Tensor] = {}


def stream_read(region: torch.Tensor, waves: int, streaming: bool) -> None:
    """Measurement only: ``waves`` single-wave workgroups read the whole of ``region`` (a multiple of 8 KB) once."""
    _check(region, "region")
    sink = _SINKS.get(region.device.index)
    if sink is None:
        sink = _SINKS[region.device.index] = torch.zeros(1, dtype=torch.float32, device=region.device)
    _call(load_module("ceilings"), "ifx_stream_read", (P, LL, I, I, P, P),
          region, region.numel() * region.element_size(), waves, int(streaming), sink, _stream())


def stream_copy(src: torch.Tensor, dst: torch.Tensor, waves: int, streaming: bool) -> None:
    """Measurement only: copies ``src`` to ``dst`` (same size, a multiple of 8 KB) with ``waves`` single-wave workgroups."""
    _check(src, "src")
    _check(dst, "dst")
    n = src.numel() * src.element_size()
    if n != dst.numel() * dst.element_size():
        raise KernelError(f"stream_copy: {n} bytes into {dst.numel() * dst.element_size()}")
    _call(load_module("ceilings"), "ifx_stream_copy", (P, P, LL, I, I, P), src, dst, n, waves, int(streaming), _stream())
