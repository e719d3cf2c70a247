"""Refresh of the MLA absorbed weights after ``kv_b_proj`` has been refitted.

``W_UV`` and ``W_UK_T`` are values derived from ``kv_b_proj`` and cached as bare module
attributes; serving graphs hold their addresses, so they are rewritten in place
(modelexpress_rl/inference/engines/vllm/installer.py:251-285;
modelexpress/engines/vllm/refit/receiver.py:229-261).  The reference computes

    kv_b = kv_b_proj.weight.view(num_heads, qk_nope_head_dim + v_head_dim, -1)
    w_uk, w_uv = kv_b.split([qk_nope_head_dim, v_head_dim], dim=1)
    W_UV.copy_(w_uv.transpose(0, 1).to(out_dtype))
    W_UK_T.copy_(w_uk.permute(1, 2, 0).to(out_dtype))

Here both are strided views of ``kv_b_proj.weight`` handed to the engine: ``W_UV`` keeps the
innermost dimension (a row gather), ``W_UK_T`` is a true transpose (the LDS transpose kernel),
each converting to the attribute's dtype on the way, with no intermediate tensor; all layers
of the model go out in one call.
"""

from __future__ import annotations

import ctypes as C
import sys
from array import array
from typing import Any

from . import _lib as L
from .engine import CAST_CODES, PlacementEngine, _put_view, _view_words, _views_of
from .load_strategy import safetensors_dtype_of


class IncompleteRefit(RuntimeError):
    """The refit ran and still left part of the model unwritten (refit/reshard/types.py:27-35)."""


_ABSENT = object()


def update_mla_absorbed_weights(engine: PlacementEngine, model: Any, *, quantized: bool, stream: int = 0) -> int:
    """Recomputes ``W_UV`` / ``W_UK_T`` of every MLA module of ``model`` in place; returns how many
    tensors were rewritten.  A no-op for models without MLA.  ``quantized``: the live ``kv_b_proj`` is
    stored quantized - its values are not the weights, so the refresh is refused as the reference does."""
    casts = {}
    native = None if quantized else L.tensors()
    words = None if native is None else native.mla_views(model, sys.modules["torch"].nn.Module, lambda m: _views_of_module(m, False, casts))
    if words is None:  # not a plain tree of modules, or something to refuse
        words = _views_of_modules(model, quantized)
    n = len(words) * getattr(words, "itemsize", 1) // C.sizeof(L.ViewCopy)
    if n:
        engine.copy_views_array(_views_of(words, n), n, stream=stream)
    return n


def _views_of_modules(model: Any, quantized: bool):
    """The words of the views, module by module; ``mla_views`` of csrc/mxp_tensors.cpp is its quick half."""
    words, casts = array("q"), {}
    for _name, module in model.named_modules():
        words += _views_of_module(module, quantized, casts)
    return words


def _views_of_module(module: Any, quantized: bool, casts: dict):
    views = []
    if not hasattr(module, "kv_b_proj"):
        return array("q")
    w_uv, w_uk_t = getattr(module, "W_UV", _ABSENT), getattr(module, "W_UK_T", _ABSENT)
    if w_uv is _ABSENT and w_uk_t is _ABSENT:
        return array("q")
    if quantized:
        raise IncompleteRefit("MLA derived-weight refresh from a quantized kv_b_proj is unsupported")
    w = module.kv_b_proj.weight
    heads, nope, v_dim = int(module.num_heads), int(module.qk_nope_head_dim), int(module.v_head_dim)
    w_shape = tuple(w.shape)
    if len(w_shape) != 2 or not w.is_contiguous() or w_shape[0] != heads * (nope + v_dim):
        raise IncompleteRefit(f"kv_b_proj.weight of shape {w_shape} does not hold {heads} heads of {nope} + {v_dim} rows")
    latent = w_shape[1]
    head_stride = (nope + v_dim) * latent
    src, es, src_type = w.data_ptr(), w.element_size(), w.dtype
    # (attribute, view shape, source strides of that view in elements, first source element)
    for attr, out, shape, strides, first in (
            ("W_UV", w_uv, (v_dim, heads, latent), (latent, head_stride, 1), nope * latent),
            ("W_UK_T", w_uk_t, (nope, latent, heads), (latent, 1, head_stride), 0)):
        if out is None or out is _ABSENT:
            continue
        if out.shape != shape:
            raise IncompleteRefit(f"{attr} has shape {tuple(out.shape)}, the view of kv_b_proj is {shape}")
        cast = casts.get((src_type, out.dtype))
        if cast is None:
            src_dtype, dst_dtype, cast = safetensors_dtype_of(w), safetensors_dtype_of(out), 0
            if dst_dtype != src_dtype:
                cast = CAST_CODES.get((src_dtype, dst_dtype), 0)
                if not cast:
                    raise IncompleteRefit(f"{attr}: no conversion from {src_dtype} to {dst_dtype}")
            casts[src_type, out.dtype] = cast
        views.append((src + first * es, out.data_ptr(), out.element_size(), cast, shape, strides, out.stride()))
    words = _view_words(len(views)) if views else array("q")
    for k, view in enumerate(views):
        _put_view(words, k, *view)
    return words
