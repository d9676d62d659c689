"""Block-sparse attention operators on one MI355X: forward, backward, merge of partials.

Host side of the C ABI in ``include/ultraattn.h``.  Tensors follow the reference's tile
kernel (``orchestrated_attn/orchestrated_attn_impl.py:326`` comment): q, o, do, dq
``[B, Sq, Nh, 128]`` bf16; k, v, dk, dv ``[B, Skv, Nh, 128]`` bf16; lse, delta ``[B, Nh, Sq]``
fp32.  Everything runs on the current CUDA(HIP) stream; nothing synchronises.
"""
from typing import Optional, Sequence, Tuple, Union

import numpy as np
import torch

from ._lib import native
from .tilelist import TILE, TileList, prepared_mask

HEAD_DIM = 128


def _tiles_for(tiles: Union[TileList, np.ndarray, torch.Tensor], q, block, causal, q_block_offset):
    """(device lists, query tiles, key tiles, active tiles) of a tile list or a block mask on q's device."""
    if not q.is_cuda:
        raise ValueError("q must be a CUDA (HIP) tensor")
    if not isinstance(tiles, TileList):
        if isinstance(tiles, torch.Tensor):
            tiles = tiles.cpu().numpy()
        m = np.asarray(tiles)
        if block is None:
            if q.shape[1] % m.shape[0] != 0:
                raise ValueError("cannot infer block size: Sq is not a multiple of the mask's rows")
            block = q.shape[1] // m.shape[0]
        m = prepared_mask(m, block, causal, q_block_offset)
        return native().lists_from_mask(m, m.shape[0], m.shape[1], block // TILE, q.device.index)
    return tiles.packed(q.device), tiles.n_qtiles, tiles.n_ktiles, tiles.nnz


def bsa_fwd(q, k, v, tiles, softmax_scale: Optional[float] = None, causal: bool = False,
            q_block_offset: int = 0, out: Optional[torch.Tensor] = None, block: Optional[int] = None,
            lse: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Block-sparse flash-attention forward -> (out, lse).

    ``tiles`` is a ``TileList`` or a block mask (0/1/2 or bool; ``causal`` and
    ``q_block_offset`` then apply the executor's diagonal rule).  One launch replaces the
    per-rectangle ``_flash_attn_forward`` calls of ``fwd_comp_func``
    (``orchestrated_attn/orchestrated_attn_impl.py:320-338``).  ``out`` is written in place
    when given (the fork's ``out=`` argument)."""
    return native().bsa_forward(q, k, v, *_tiles_for(tiles, q, block, causal, q_block_offset), softmax_scale, out, lse)


def softmax_delta(out, dout, delta: Optional[torch.Tensor] = None) -> torch.Tensor:
    """delta = rowsum(dout * out) as fp32 [B, Nh, Sq]: the ``softmax_d`` input of the fork's
    backward (``orchestrated_attn/orchestrated_attn_impl.py:595``)."""
    return native().delta(out, dout, delta)


def bsa_bwd(dout, q, k, v, out, lse, tiles, softmax_scale: Optional[float] = None, causal: bool = False,
            dq=None, dk=None, dv=None, softmax_d: Optional[torch.Tensor] = None, q_block_offset: int = 0,
            block: Optional[int] = None) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Block-sparse backward -> (dq, dk, dv), written in place when the buffers are given
    (as ``_flash_attn_backward`` does, ``orchestrated_attn/orchestrated_attn_impl.py:578-596``).
    ``lse`` (and ``softmax_d`` when given; then ``out`` is ignored and may be None, the
    reference passes a dummy) are the rows' global statistics."""
    return native().bsa_backward(dout, q, k, v, out, lse, dq, dk, dv, softmax_d,
                                 *_tiles_for(tiles, q, block, causal, q_block_offset), softmax_scale)


def merge_partials(outs: Sequence[torch.Tensor], lses: Sequence[torch.Tensor],
                   out: Optional[torch.Tensor] = None, lse: Optional[torch.Tensor] = None):
    """LSE-weighted merge of partial outputs -> (out, lse): one pass in place of the chain of
    ``update_out_and_lse`` calls (``ring_flash_attn/utils.py:38-52, 78-99``).
    outs[p]: contiguous [B, S, Nh, 128] bf16; lses[p]: contiguous [B, Nh, S] fp32."""
    return native().merge(outs, lses, out, lse)


def grad_accumulate(partial: torch.Tensor, out: Optional[torch.Tensor], acc: Optional[torch.Tensor] = None,
                    init_from_out: bool = False) -> None:
    """One step of the gradient accumulation that the reference specifies
    (``ring_flash_attn/ring_flash_attn.py:110-118``) and its packs leave as stubs
    (``orchestrated_attn/utils.py:260-262, 296-298``), as one kernel (``ua_grad_accumulate``):

    * ``acc`` (fp32) given: ``acc += partial`` and ``out = bf16(acc)`` (``out`` may be None);
      with ``init_from_out`` the sum starts from ``out``: ``acc = float(out) + partial``;
    * no ``acc``: ``out = bf16(float(out) + partial)``.
    ``partial`` and ``out`` are contiguous bf16 tensors of equal size, ``acc`` contiguous fp32."""
    native().grad_accumulate(partial, out, acc, init_from_out)


def grad_sum(parts: Sequence[torch.Tensor], out: Optional[torch.Tensor] = None, scale: float = 1.0) -> torch.Tensor:
    """``out = bf16(scale * sum(parts))`` with the sum carried in fp32, one pass (``ua_grad_sum``).
    parts: 1..16 contiguous ``[B, S, Nh, 128]`` tensors, all bf16 or all fp32; ``out`` bf16, may be a
    strided view (head_dim contiguous)."""
    return native().grad_sum(parts, out, scale)


def update_out_and_lse(out: Optional[torch.Tensor], lse: Optional[torch.Tensor], block_out: torch.Tensor,
                       block_lse: torch.Tensor, slice_=None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Drop-in for ``update_out_and_lse`` of the ring / hierarchy executors
    (``ring_flash_attn/utils.py:78-99``; call sites ``hierarchy_attn/hierarchy_attn_impl.py:64-81``):
    folds one more partial ``(block_out [B,Sb,Nh,D], block_lse [B,Nh,Sb])`` into the running
    ``(out [B,S,Nh,D], lse [B,S,Nh,1])`` and returns the pair.

    * first call (``out is None``): returns ``block_out`` and ``block_lse`` as ``[B,S,Nh,1]``, as the
      reference does (``slice_`` is then an error);
    * ``slice_`` (an index for both ``out`` and ``lse``, e.g. ``(slice(None), slice(S//2, None))``):
      the rows it selects are updated in place, in ``out``'s dtype;
    * otherwise new tensors are returned and ``out`` is fp32, which is what the reference's
      expression yields (fp32 statistics times bf16 rows).
    One kernel (``ua_merge_update``) in place of the reference's eight element-wise launches; the
    arithmetic is max-stabilised and treats ``lse = -inf`` as "no keys", which the literal formula
    does not (it agrees with it on every input where that one is finite).  ``block_lse`` may also
    come as ``[B,Sb,Nh,1]`` (the hierarchy executor's ``forward`` closure, ``:40-53``)."""
    if out is None:
        if slice_ is not None:
            raise RuntimeError("first update_out_and_lse should not pass slice_ args")
        if block_lse.dim() == 3:
            block_lse = block_lse.transpose(-2, -1).unsqueeze(dim=-1)
        return block_out, block_lse
    if slice_ is None:
        return native().merge_update(out, lse, block_out, block_lse, False)
    tgt_out, tgt_lse = out[slice_], lse[slice_]
    if tgt_out.untyped_storage().data_ptr() != out.untyped_storage().data_ptr() or \
            tgt_lse.untyped_storage().data_ptr() != lse.untyped_storage().data_ptr():
        # the reference assigns `out[slice_] = ...`, which writes through any index; a kernel can
        # only write through a view
        raise ValueError("slice_ must select a view of out and lse (slices, not index lists or tensors)")
    native().merge_update(tgt_out, tgt_lse, block_out, block_lse, True)
    return out, lse
