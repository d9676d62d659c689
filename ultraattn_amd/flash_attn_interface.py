"""Drop-in for the two functions the reference's executors import from the flash-attention
fork: ``from flash_attn.flash_attn_interface import _flash_attn_forward, _flash_attn_backward``
(``orchestrated_attn/orchestrated_attn_impl.py:7-8``, ``hierarchy_attn/hierarchy_attn_impl.py:3``).

Same positional/keyword arguments, including the fork's ``out=`` (forward) and ``softmax_d=``
(backward).  A call is one dense rectangle: it goes to ``ua_dense_fwd`` / ``ua_dense_bwd``, which
enumerate the tiles themselves (no tile list is built, copied or cached) and cut rectangles with
few tile lines into parts that fill the device.  Nothing here synchronises or copies from the
host, so a call (a first call at a new shape included) can be captured into a HIP graph.
"""
from typing import Dict, Optional, Tuple

import torch

from ._lib import native

# (device index, stream handle) -> uint8 tensor holding the partial results of split calls.  Calls
# on one stream run in order, so they can share it; it only ever grows, and the native side keeps
# a bounded number of them (least recently used first out: stream handles come and go).
_workspaces: Dict[Tuple[int, int], torch.Tensor] = {}
_captured = []             # workspaces that a captured graph may replay into: never released
_NO_WINDOW = (-1, -1)


def _check_unsupported(dropout_p, window_size, alibi_slopes, return_softmax=False):
    if dropout_p != 0:
        raise NotImplementedError("dropout_p must be 0")
    if tuple(window_size) != (-1, -1):
        raise NotImplementedError("window_size must be (-1, -1)")
    if alibi_slopes is not None:
        raise NotImplementedError("alibi_slopes must be None")
    if return_softmax:
        raise NotImplementedError("return_softmax needs dropout_p > 0, which is unsupported")


def _flash_attn_forward(q, k, v, dropout_p, softmax_scale, causal, window_size=(-1, -1),
                        alibi_slopes=None, return_softmax=False, out=None):
    """-> (out, q, k, v, out_padded, softmax_lse, S_dmask, rng_state); callers use [0] and [5]
    (``orchestrated_attn_impl.py:326``, ``hierarchy_attn_impl.py:41``).  With ``causal`` and
    Sq != Skv the diagonal is aligned to the bottom-right corner, as flash-attn (2.1 and later)
    does: query i sees key j iff j <= i + Skv - Sq."""
    if dropout_p != 0 or window_size != _NO_WINDOW or alibi_slopes is not None or return_softmax:
        _check_unsupported(dropout_p, window_size, alibi_slopes, return_softmax)
    out, lse = native().dense_forward(q, k, v, softmax_scale, causal, out, _workspaces, _captured)
    return out, q, k, v, out, lse, None, None


def _flash_attn_backward(dout, q, k, v, out, softmax_lse, dq, dk, dv, dropout_p, softmax_scale, causal,
                         window_size=(-1, -1), alibi_slopes=None, deterministic=False, rng_state=None,
                         softmax_d: Optional[torch.Tensor] = None):
    """Writes dq, dk, dv in place (allocates the ones passed as None); returns (dq, dk, dv, softmax_d).  With ``softmax_d`` given
    ``out`` is ignored (the reference passes a dummy, ``orchestrated_attn_impl.py:583``).
    The kernels are deterministic regardless of ``deterministic``."""
    if dropout_p != 0 or window_size != _NO_WINDOW or alibi_slopes is not None:
        _check_unsupported(dropout_p, window_size, alibi_slopes)
    return native().dense_backward(dout, q, k, v, out, softmax_lse, dq, dk, dv, softmax_d, softmax_scale, causal, _workspaces, _captured)
