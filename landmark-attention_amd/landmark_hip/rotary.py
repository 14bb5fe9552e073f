"""Rotary position embedding on the HIP kernel, with the reference's call surface.

``apply_rotary_pos_emb(q, k, cos, sin, position_ids)`` mirrors ``llama/llama_mem.py:134-149``:
``cos``/``sin`` are the ``(1, 1, n_pos, hd)`` (or ``(n_pos, hd)``) model-dtype tables of
``LlamaRotaryEmbedding`` (``:95-124``), ``position_ids`` is ``(bs, seq)`` or ``(1, seq)`` int64, ``q`` may
be ``None`` (``:143-144``).  One launch for q and k together (one per tensor when their shapes differ) replaces the reference's gather of the table rows,
two products, ``rotate_half``'s concatenation and the sum, and gives the same bits: every one of the
three elementwise operations rounds to the model dtype, as torch's 16-bit arithmetic does.
"""
from __future__ import annotations

import torch

from . import _lib


def _transposed_sin(sin):
    """The sine table of the transposed rotation.  ``y = x*cos + rotate_half(x)*sin`` is linear in x, and its
    transpose is the same expression with ``sin`` replaced by ``-cat(sin[..., hd/2:], sin[..., :hd/2])``
    (for LLaMA's tables, whose halves are equal, simply ``-sin``: the rotation by the opposite angle).  The
    gradient therefore goes through the same kernel, with the same three roundings torch's autograd applies
    to the reference expression in a 16-bit model."""
    h = sin.shape[-1] // 2
    return (-torch.cat((sin[..., h:], sin[..., :h]), dim=-1)).contiguous()


class _Rotary(torch.autograd.Function):
    """The rotation of one tensor as an operation torch can record; the backward is the transposed rotation."""

    @staticmethod
    def forward(ctx, x, cos, sin, position_ids):
        ctx.save_for_backward(cos, sin, position_ids)
        return _lib.native().rotate(x, cos, sin, position_ids)

    @staticmethod
    def backward(ctx, dy):
        cos, sin, position_ids = ctx.saved_tensors
        return _lib.native().rotate(dy, cos, _transposed_sin(sin), position_ids), None, None, None


def apply_rotary_pos_emb(q, k, cos, sin, position_ids):
    """``(q_embed, k_embed)`` as ``llama_mem.py:134-149`` returns them; ``q_embed`` is ``None`` when
    ``q`` is.  q, k: ``(B, nh, L, hd)`` bf16/fp16 on the GPU with hd 64 or 128.  Differentiable in q and k,
    as the reference's expression is (the tables and positions get no gradient): the backward is the transposed
    rotation (``_transposed_sin``), for which the kernel reads the sine table in place."""
    if q is not None and q.shape != k.shape:    # e.g. fewer key heads: one launch per tensor
        return tuple(apply_rotary_pos_emb(None, x, cos, sin, position_ids)[1] for x in (q, k))
    rotated = _lib.native().rotary(q, k, cos, sin, position_ids)
    if rotated is not None:
        return rotated
    # under torch.jit.trace, which records a Function (one per tensor) as an operation, or with forward-mode gradients, which
    # it refuses
    return None if q is None else _Rotary.apply(q, cos, sin, position_ids), _Rotary.apply(k, cos, sin, position_ids)
