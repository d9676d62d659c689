"""What a row's result depends on: over a tile list on its own list alone, so that a launch over one head, or over some of
the rows or columns of a mask, gives bit for bit what the whole gives; a dense rectangle without a workspace equals
its tile list.  Launches on both sides of the sizes at which dense rectangles change their workgroups."""
import numpy as np
import pytest
import torch

from tests.gpu_util import SCALE
from tests.test_gpu_dense import dense_unsplit
from ultraattn_amd import masks, ops
from ultraattn_amd.tilelist import build_tile_list

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(sq, sk, nh, batch=1):
    g = torch.Generator(device=DEV).manual_seed(sq + nh)
    mk = lambda n: torch.randn(batch, n, nh, 128, device=DEV, generator=g).to(torch.bfloat16)
    return mk(sq), mk(sk), mk(sk), mk(sq)


@pytest.mark.parametrize("mask,nh", [
    (masks.config_strided(16, 2, 4), 40),              # 640 rows: one head has 16, half the rows 320
    (masks.config_causal(24), 24),                     # 576, 24, 288
    (masks.config_global_local(32), 8),                # 256, 32, 128
    (masks.config_streaming_shard(6, 40, 5), 48),      # 288 rows and 1920 columns
])
def test_heads_and_shards(mask, nh):
    n = mask.shape[0]
    q, k, v, do = _inputs(n * 128, mask.shape[1] * 128, nh)
    o, lse = ops.bsa_fwd(q, k, v, mask, SCALE, block=128)
    delta = ops.softmax_delta(o, do)
    bwd = lambda *a, **kw: ops.bsa_bwd(*a[:4], None, *a[4:], SCALE, block=128, **kw)
    dq, dk, dv = bwd(do, q, k, v, lse, mask, softmax_d=delta)
    for h in (0, nh - 1):
        s = slice(h, h + 1)
        qh, kh, vh, doh = (t[:, :, s].contiguous() for t in (q, k, v, do))
        oh, lh = ops.bsa_fwd(qh, kh, vh, mask, SCALE, block=128)
        assert torch.equal(oh, o[:, :, s]) and torch.equal(lh, lse[:, s])
        got = bwd(doh, qh, kh, vh, lse[:, s].contiguous(), mask, softmax_d=delta[:, s].contiguous())
        for a, b in zip(got, (dq, dk, dv)):
            assert torch.equal(a, b[:, :, s])
    # half the rows: the outputs of rows; half the columns: those of columns
    rows = slice(n // 2 * 128, None)
    oh, lh = ops.bsa_fwd(q[:, rows], k, v, mask[n // 2:], SCALE, block=128)
    assert torch.equal(oh, o[:, rows]) and torch.equal(lh, lse[:, :, rows])
    part = bwd(do[:, rows], q[:, rows], k, v, lse[:, :, rows].contiguous(), mask[n // 2:], softmax_d=delta[:, :, rows].contiguous())
    assert torch.equal(part[0], dq[:, rows])
    cols = slice(0, mask.shape[1] // 2 * 128)
    part = bwd(do, q, k[:, cols], v[:, cols], lse, np.ascontiguousarray(mask[:, :mask.shape[1] // 2]), softmax_d=delta)
    assert torch.equal(part[1], dk[:, cols]) and torch.equal(part[2], dv[:, cols])


@pytest.mark.parametrize("nq,nk,nh,causal", [
    (2, 2, 1, True), (3, 9, 5, False), (16, 16, 16, True), (20, 16, 10, True), (16, 20, 20, True), (8, 8, 33, False), (16, 4, 33, False),
])
def test_dense_without_workspace_equals_the_tile_list(lib, nq, nk, nh, causal):
    mask = np.ones((nq, nk), np.uint8)
    if causal:
        i, j = np.arange(nq)[:, None] + nk - nq, np.arange(nk)[None, :]
        mask = np.where(j < i, 1, np.where(j == i, 2, 0)).astype(np.uint8)
    q, k, v, do = _inputs(nq * 128, nk * 128, nh)
    o, lse = ops.bsa_fwd(q, k, v, mask, SCALE, block=128)
    delta = ops.softmax_delta(o, do)
    got = dense_unsplit(lib, q, k, v, do, causal)
    for a, b in zip((o, lse, delta, *ops.bsa_bwd(do, q, k, v, None, lse, mask, SCALE, block=128, softmax_d=delta)), got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("heads", [128, 132])                # 32768 and 33792 lines
def test_backward_of_32768_lines_and_more(heads):
    tiles = build_tile_list(masks.config_strided(16), block=512)
    q, k, v, do = _inputs(8192, 8192, heads, batch=2)
    o, lse = ops.bsa_fwd(q, k, v, tiles, SCALE)
    grads = ops.bsa_bwd(do, q, k, v, o, lse, tiles, SCALE)
    for b, h in ((0, 0), (1, heads - 1)):
        at = (slice(b, b + 1), slice(None), slice(h, h + 1))
        alone = ops.bsa_bwd(*(t[at].contiguous() for t in (do, q, k, v, o)), lse[b:b + 1, h:h + 1].contiguous(), tiles, SCALE)
        for whole, one in zip(grads, alone):
            assert torch.equal(whole[at], one)
