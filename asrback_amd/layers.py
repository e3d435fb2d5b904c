"""The element-wise work around the attention calls, as kernels of
``libasrattn.so`` (``csrc/layers.hpp``).

Each function here computes what a sequence of PyTorch ops in the model
modules computes, in fewer passes over memory, and each has a ``..._takes``
predicate: the modules call it on the tensors it takes (plain ROCm tensors
that need no gradient, in the layouts the kernels address) and run the ops
otherwise.
"""

from __future__ import annotations

import ctypes
import math

import torch
from torch import Tensor, nn
from torch.nn.modules import module as _module

from . import _lib
from .attention import _DTYPES, _stream

_VECTOR = 16  # bytes per lane access
_increment_version = torch.autograd.graph.increment_version


def _plain(*tensors: Tensor) -> bool:
    """Whether the kernels may read these tensors in place of PyTorch ops:
    ordinary ROCm tensors of one supported dtype, on the current device, with
    nothing (autograd, forward-mode, autocast, functorch, function and
    dispatch modes, tracing) that has to see the ops."""
    first = tensors[0]
    dtype, index = first.dtype, first.get_device()
    if dtype not in _DTYPES or not first.is_cuda or index != torch.cuda.current_device():
        return False
    grad = torch.is_grad_enabled()
    for t in tensors:
        if type(t) is not Tensor and type(t) is not nn.Parameter:
            return False
        if t.dtype != dtype or t.get_device() != index or (grad and t.requires_grad):
            return False
    return not (torch.is_autocast_enabled("cuda") or torch.compiler.is_compiling() or torch.jit.is_tracing()
                or torch.autograd.forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack()
                or torch._C._len_torch_function_stack() or torch._C._functorch.maybe_current_level() is not None)


def _vectors(t: Tensor) -> bool:
    """Whether rows of ``t`` (its last axis) can be read 16 bytes at a time."""
    *strides, last = t.stride()
    bits = 0
    for stride in strides:
        bits |= stride  # a vector is a power of two of elements: one test for all
    return last == 1 and t.data_ptr() % _VECTOR == 0 and bits % (_VECTOR // t.element_size()) == 0


_CALL = nn.Module.__call__
# What the kernels compute in place of a call: each class's own forward.
_FORWARDS = {c: c.forward for c in (nn.Linear, nn.LayerNorm, nn.Embedding)}


def computes(cls: type) -> type:
    """Class decorator: the kernels compute what ``cls.forward`` is now."""
    _FORWARDS[cls] = cls.forward
    return cls


def unhooked(*modules: nn.Module) -> bool:
    """Whether a call of each module is its class's own ``forward`` and nothing
    else: no hooks, and none of it replaced on the module or the class."""
    if _module._global_forward_hooks or _module._global_forward_pre_hooks or nn.Module.__call__ is not _CALL:
        return False
    seen = None
    for m in modules:
        own, cls = m.__dict__, type(m)
        if own["_forward_hooks"] or own["_forward_pre_hooks"] or "forward" in own:
            return False
        if cls is not seen:
            if cls.forward is not _FORWARDS.get(cls):
                return False
            seen = cls
    return True


def _strides(t: Tensor) -> tuple[int, int, int]:
    """Batch, token and head strides of ``(batch, tokens, heads, head_dim)``
    or ``(tokens, heads, head_dim)`` rows."""
    strides = t.stride()
    return strides[:3] if len(strides) == 4 else (0, *strides[:2])


def prompt_rows_takes(q: Tensor, k: Tensor | None, v: Tensor | None, k_cache, v_cache, rows: Tensor | None,
                      positions: Tensor | None, q_norm: nn.Module, k_norm: nn.Module | None, cos: Tensor,
                      sin: Tensor) -> bool:
    """Whether :func:`prompt_rows` takes these (see there): rows ``q``
    ``(batch, tokens, heads, head_dim)`` or ``(tokens, heads, head_dim)``,
    tables ``(batch, tokens, head_dim)`` or ``(tokens, head_dim)``, caches
    ``(rows, length, heads, head_dim)``."""
    norms = [q_norm] if k_norm is None else [q_norm, k_norm]
    weights = [m.weight for m in norms]
    tensors = [q, cos, sin, *weights]
    if k is not None:
        tensors += [k, v, k_cache, v_cache]
    if not _plain(*tensors) or not unhooked(*norms):
        return False
    *batch, tokens, _, head_dim = q.shape
    if head_dim not in (64, 128, 256, 512) or any(w.shape != (head_dim,) for w in weights):
        return False
    if cos.shape != sin.shape or cos.stride() != sin.stride() or cos.shape[-2:] != (tokens, head_dim):
        return False
    if cos.dim() > q.dim() - 1 or (cos.dim() == 3 and cos.shape[0] not in (1, *batch)):
        return False
    if k is not None:
        slots = (math.prod(batch) * tokens if positions is not None else math.prod(batch),)
        for index in (rows, positions):
            if index is None:
                continue
            if (type(index) is not Tensor or index.dtype != torch.int64 or index.shape != slots
                    or index.device != q.device or not index.is_contiguous()):
                return False
        if positions is None and tokens > k_cache.shape[1]:
            return False
        if not torch.is_inference_mode_enabled() and (k_cache.is_inference() or v_cache.is_inference()):
            return False  # the ops refuse the write
        if (k.shape != v.shape or k_cache.shape != v_cache.shape or k_cache.dim() != 4
                or k_cache.shape[2:] != k.shape[-2:] or k.shape[-1] != head_dim):
            return False
    return all(_vectors(t) for t in tensors)


def prompt_rows(q: Tensor, k: Tensor | None, v: Tensor | None, k_cache: Tensor | None, v_cache: Tensor | None,
                rows: Tensor | None, positions: Tensor | None, q_norm: nn.Module, k_norm: nn.Module | None, cos: Tensor,
                sin: Tensor, *, block_table: Tensor | None = None, v_eps: float | None = None):
    """What a prompt pass does to its projections before the attention
    (``asrlayer_prompt_rows``; ``qwen3_asr.py:366-390``, ``gemma4.py:515-561``):
    the per-head norms and the rotation of ``q`` and ``k`` ``(batch, tokens,
    heads, head_dim)`` (no batch: one), with ``v_eps`` the weightless norm of ``v``, and the
    writes of keys and values to the cache at ``(rows, positions)``, int64 per
    token, or, without ``positions``, at tokens ``0 .. tokens - 1`` of
    ``rows[b]``.  With ``block_table`` the caches are page pools whose last
    page takes what no row owns.  Returns contiguous ``q``, ``k`` and ``v``
    (``v`` itself where it is not normalized); ``k`` None: ``q`` alone."""
    tokens, heads, head_dim = q.shape[-3:]
    batch = q.shape[0] if q.dim() == 4 else 1
    q_out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    rope = (cos.stride(0) if cos.dim() == 3 and cos.shape[0] > 1 else 0, cos.stride(-2))
    common = (q_norm.weight.data_ptr(), None if k is None else k_norm.weight.data_ptr(), cos.data_ptr(), sin.data_ptr(),
              *rope, q_norm.eps, 0.0 if k is None else k_norm.eps, v_eps or 0.0, v_eps is not None, batch, tokens,
              heads)
    if k is None:
        params = _lib.PromptParams(
            q.data_ptr(), None, None, q_out.data_ptr(), None, None, None, None, *_strides(q), *(0,) * 12, 0, 0,
            None, None, None, 0, 0, 0, *common, 0, head_dim, _DTYPES[q.dtype])
        k_out = v_out = None
    else:
        k_out = torch.empty(k.shape, dtype=q.dtype, device=q.device)
        v_out = v if v_eps is None else torch.empty(v.shape, dtype=q.dtype, device=q.device)
        if block_table is None:
            extent = (k_cache.shape[0], k_cache.shape[1])
            table = (None, 0, 0, 0)
        else:
            extent = (block_table.shape[0], 0)
            table = (block_table.data_ptr(), block_table.shape[1], k_cache.shape[1], k_cache.shape[0] - 1)
        params = _lib.PromptParams(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), q_out.data_ptr(), k_out.data_ptr(),
            None if v_eps is None else v_out.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
            *_strides(q), *_strides(k), *_strides(v), *_strides(k_cache), *_strides(v_cache), *extent,
            rows.data_ptr(), None if positions is None else positions.data_ptr(), *table, *common, k.shape[-2], head_dim,
            _DTYPES[q.dtype])
    lib = _lib.load()
    _lib.check(lib.asrlayer_prompt_rows(ctypes.byref(params), _stream(q.device)), "asrlayer_prompt_rows")
    if k is not None:
        _increment_version((k_cache, v_cache))
    return q_out, k_out, v_out


# Rows a decoder step's linear layers take (csrc/rows_linear.hip), and in bf16
# with a reduction of more than 4096 inputs among them (whole decoder layers
# against the ops, 64 encoder frames: bf16, width 1280, fc2 of 5120 inputs, 8 rows
# 66 us and 90, 12 rows 83 and 93, 13 to 16 101 and 85-92; width 1024, 16 rows 62
# and 81; float32, width 768, 16 rows 52 and 87, 1024, 12 rows 71 and 96).
LINEAR_ROWS, LONG_LINEAR_ROWS = 16, 12


def rows_linear_takes(x: Tensor, linears: list[nn.Module], norms: list[nn.Module], wide: list[nn.Module]) -> bool:
    """Whether :func:`rows_linear` takes ``x`` ``(rows, 1, inputs)`` through
    each of ``linears`` and ``norms``, and ``(rows, 1, outputs)`` of the last of
    ``linears`` through each of ``wide``."""
    modules = [*linears, *wide, *norms]
    if any(type(m) is not nn.Linear for m in (*linears, *wide)) or any(type(m) is not nn.LayerNorm for m in norms):
        return False
    held = [(m.weight, m.bias) for m in modules]  # each looked up once
    tensors = [x]
    for weight, bias in held:
        tensors += [weight] if bias is None else [weight, bias]
    if any(t is None for t in tensors) or not _plain(*tensors) or not unhooked(*modules):
        return False
    if x.dim() != 3 or x.shape[1] != 1 or not 1 <= x.shape[0] <= LINEAR_ROWS or not _vectors(x[:, 0]):
        return False
    inputs, per = x.shape[2], _VECTOR // x.element_size()
    last = len(linears)
    if any(weight.dim() != 2 for weight, _ in held[:last + len(wide)]):
        return False
    for width, layers in ((inputs, held[:last]), (held[last - 1][0].shape[0], held[last:last + len(wide)])):
        if not layers:
            continue
        if width % per or not 0 < width // per <= 1024 or (per == 8 and width > 4096 and x.shape[0] > LONG_LINEAR_ROWS):
            return False
        for weight, bias in layers:
            if weight.shape[1] != width or not weight.is_contiguous() or not _vectors(weight):
                return False
            if bias is not None and (bias.shape != weight.shape[:1] or not bias.is_contiguous()):
                return False
    return all(m.normalized_shape == weight.shape == (inputs,) and bias is not None and bias.shape == weight.shape
               and _vectors(weight) and _vectors(bias) for m, (weight, bias) in zip(norms, held[last + len(wide):]))


def rows_linear(x: Tensor, linears: list[nn.Linear], norm: nn.LayerNorm | None = None, *, gelu: bool = False,
                residual: Tensor | None = None) -> list[Tensor]:
    """``[linear(norm(x)) for linear in linears]`` for a decoder step's few
    rows, in one launch (``asrlayer_rows_linear``): up to three matrices, with
    ``gelu`` (exact) after them or, with one matrix, ``residual`` ``(rows, 1,
    outputs)`` of unit last stride added to the result."""
    rows, _, inputs = x.shape
    weights = [m.weight for m in linears]
    outs = [torch.empty((rows, 1, w.shape[0]), dtype=x.dtype, device=x.device) for w in weights]
    if residual is not None and (residual.shape != outs[0].shape or residual.stride(2) != 1):
        raise ValueError(f"a residual of {tuple(residual.shape)} for {rows} rows of {outs[0].shape[2]}")
    params = _lib.LinearParams()
    params.x, params.x_row_stride = x.data_ptr(), x.stride(0)
    if norm is not None:
        params.ln_weight, params.ln_bias, params.ln_eps = norm.weight.data_ptr(), norm.bias.data_ptr(), norm.eps
    for i, (m, weight, out) in enumerate(zip(linears, weights, outs)):
        params.w[i], params.out[i], params.n[i] = weight.data_ptr(), out.data_ptr(), weight.shape[0]
        bias = m.bias
        if bias is not None:
            params.b[i] = bias.data_ptr()
    if residual is not None:
        params.residual, params.r_row_stride = residual.data_ptr(), residual.stride(0)
    params.rows, params.k, params.act, params.dtype = rows, inputs, int(gelu), _DTYPES[x.dtype]
    lib = _lib.load()
    _lib.check(lib.asrlayer_rows_linear(ctypes.byref(params), _stream(x.device)), "asrlayer_rows_linear")
    return outs


# A vocabulary product (51865 outputs) takes up to two rows, and more of the
# short ones: float rows of 768, 1: 46.2 -> 30.6 us, 3: 28.1 -> 25.6, 4: 36.0 ->
# 32.0; of 1280, 1: 72.4 -> 46.5, 4: 53.7 -> 55.9; bf16 rows of 384, 4: 13.2 ->
# 10.1, of 512, 4: 13.8 -> 11.5, of 768, 3: 16.5 -> 17.1, of 1280, 2: 23.4 -> 23.2
# (of 640, a width that no Whisper has, 4: 14.6 -> 16.4).
# Float rows' worst error against float64 is 5 times smaller (sums of vectors,
# then trees).
PRODUCT_ROWS, PRODUCT_VALUES, PRODUCT_INPUTS_BF16 = 4, 2560, 640


def rows_product_takes(x: Tensor, weight: Tensor) -> bool:
    """Whether :func:`rows_product` takes ``x`` ``(rows, inputs)`` and ``weight``
    ``(outputs, inputs)``."""
    if not _plain(x, weight) or x.dim() != 2 or weight.dim() != 2 or not 1 <= x.shape[0] <= PRODUCT_ROWS:
        return False
    inputs, per = weight.shape[1], _VECTOR // x.element_size()
    if x.shape[0] > 2 and per == 8 and inputs > PRODUCT_INPUTS_BF16:
        return False
    return (x.shape[1] == inputs and 0 < x.shape[0] * inputs <= PRODUCT_VALUES and inputs % per == 0
            and inputs // per <= 384 and weight.shape[0] > 0 and _vectors(x) and weight.is_contiguous()
            and _vectors(weight))


def rows_product(x: Tensor, weight: Tensor) -> Tensor:
    """``x @ weight.T`` for a step's few rows (``asrlayer_rows_linear``)."""
    (rows, inputs), outputs = x.shape, weight.shape[0]
    out = torch.empty((rows, outputs), dtype=x.dtype, device=x.device)
    params = _lib.LinearParams()
    params.x, params.x_row_stride = x.data_ptr(), x.stride(0)
    params.w[0], params.out[0], params.n[0] = weight.data_ptr(), out.data_ptr(), outputs
    params.rows, params.k, params.dtype = rows, inputs, _DTYPES[x.dtype]
    lib = _lib.load()
    _lib.check(lib.asrlayer_rows_linear(ctypes.byref(params), _stream(x.device)), "asrlayer_rows_linear")
    return out


def embed_rows_takes(tokens: Tensor, positions: Tensor, token_table: nn.Module, position_table: nn.Module) -> bool:
    """Whether :func:`embed_rows` takes ``tokens`` ``(rows, 1)`` and
    ``positions`` ``(rows,)`` through these embeddings."""
    tables = (token_table, position_table)
    if any(type(m) is not nn.Embedding or m.max_norm is not None for m in tables) or not unhooked(*tables):
        return False
    a, b = token_table.weight, position_table.weight
    if not _plain(a, b) or a.shape[1] != b.shape[1] or a.shape[1] % (_VECTOR // a.element_size()):
        return False
    if not (a.is_contiguous() and b.is_contiguous() and _vectors(a) and _vectors(b)):
        return False
    return (type(tokens) is Tensor and type(positions) is Tensor and tokens.dtype == positions.dtype == torch.int64
            and tokens.dim() == 2 and tokens.shape[1] == 1 and positions.shape == tokens.shape[:1]
            and len(positions) > 0 and positions.is_contiguous()
            and tokens.get_device() == positions.get_device() == a.get_device())


def embed_rows(tokens: Tensor, positions: Tensor, token_table: nn.Embedding, position_table: nn.Embedding) -> Tensor:
    """``token_table(tokens) + position_table(positions)[:, None]`` for a
    decoder step, in one launch (``asrlayer_embed_rows``)."""
    a, b = token_table.weight, position_table.weight
    rows, width = tokens.shape[0], a.shape[1]
    out = torch.empty((rows, 1, width), dtype=a.dtype, device=a.device)
    params = _lib.EmbedParams(a.data_ptr(), b.data_ptr(), tokens.data_ptr(), positions.data_ptr(), out.data_ptr(),
                              tokens.stride(0), a.shape[0], b.shape[0], rows, width, _DTYPES[a.dtype])
    lib = _lib.load()
    _lib.check(lib.asrlayer_embed_rows(ctypes.byref(params), _stream(a.device)), "asrlayer_embed_rows")
    return out


def gemm_takes(x: Tensor, linear: nn.Module) -> bool:
    """Whether :func:`gemm` takes ``x`` ``(batch, rows, inputs)`` through
    ``linear`` (bf16)."""
    if type(linear) is not nn.Linear or x.dim() != 3 or x.dtype != torch.bfloat16:
        return False
    weight, bias = linear.weight, linear.bias
    shape = weight.shape
    if len(shape) != 2:
        return False
    outputs, inputs = shape
    if bias is not None and bias.numel() != outputs:
        return False
    if inputs % 64 or outputs % 8 or x.shape[2] != inputs or not unhooked(linear):
        return False
    if not (_plain(x, weight) if bias is None else _plain(x, weight, bias)):
        return False
    return (_vectors(x) and inputs <= x.stride(1) <= 1 << 22 and weight.is_contiguous() and _vectors(weight)
            and (bias is None or _vectors(bias)))


def gemm_few(x: Tensor) -> bool:
    """Whether :func:`gemm` of a square layer over ``x`` ``(batch, rows,
    inputs)`` takes no longer on the GPU than the library's product (and 10 us
    less of host time): up to 768 inputs, 256 tiles of 32 x 32 outputs (us against
    the library's: 32 rows of 768 4.2 and 5.2, 300 rows 5.6 and 5.5, 384 8.1 and
    6.0); longer rows, 256 of 16 x 16 (32 rows of 1280 5.0 and 5.5, 96 6.2 and 5.7)."""
    batch, rows, inputs = x.shape
    tile = 32 if inputs <= 768 else 16
    return -(-batch * rows // tile) * -(-inputs // tile) <= 256


def used_takes(used: Tensor, x: Tensor) -> bool:
    """Whether ``used`` can count the rows of ``x`` ``(batch, rows, inputs)``
    that :func:`gemm` computes."""
    return (type(used) is Tensor and used.dtype == torch.int32 and used.shape == x.shape[:1]
            and used.get_device() == x.get_device() and used.is_contiguous())


def gemm(x: Tensor, linear: nn.Linear, used: Tensor | None = None, into: Tensor | None = None) -> Tensor:
    """``linear(x)`` for bf16 ``x`` ``(batch, rows, inputs)``, or ``into + x
    @ linear.weight.T`` written to ``into`` (contiguous; no bias), in one
    launch (``asrlayer_gemm``).  ``used`` (int32 per batch entry): the rows that
    are computed; the others hold anything (``into``: what they held)."""
    batch, rows, inputs = x.shape
    weight = linear.weight
    outputs = weight.shape[0]
    if into is not None and (into.shape != (batch, rows, outputs) or not into.is_contiguous()):
        raise RuntimeError(f"{batch} x {rows} rows of {outputs} outputs added to a {tuple(into.shape)} tensor")
    out = into
    if into is None:
        out = torch.empty((batch, rows, outputs), dtype=x.dtype, device=x.device)
    bias = linear.bias if into is None else None
    x_strides, out_strides = x.stride()[:2], out.stride()[:2]
    if used is None and x_strides[0] == rows * x_strides[1]:
        batch, rows = 1, batch * rows  # one run of rows: fewer part-filled tiles
    params = _lib.GemmParams(
        x.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), out.data_ptr(),
        None if used is None else used.data_ptr(), *x_strides, *out_strides, batch, rows, outputs, inputs,
        into is not None)
    lib = _lib.load()
    _lib.check(lib.asrlayer_gemm(ctypes.byref(params), _stream(x.device)), "asrlayer_gemm")
    return out
