"""The backward's two sides in one launch (ua_bsa_bwd) equal the two separate launches bit for bit: the
same walks, whatever shares a CU with them.  Masks with one tile, empty lines, more columns than rows and
causal tiles; head counts on both sides of the XCD mapping; up to 256 lines on both sides together, up to 512 (where the
one launch takes the columns in reverse) and beyond."""
import numpy as np
import pytest
import torch

from tests.gpu_util import SCALE
from ultraattn_amd import _lib, masks, ops
from ultraattn_amd.tilelist import build_tile_list

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("mask,nh,batch", [
    (np.full((1, 1), 2, np.uint8), 1, 1),
    (np.zeros((2, 3), np.uint8), 3, 1),
    (masks.config_strided(9, 2, 4), 5, 2),
    (masks.config_streaming_shard(3, 11, 2), 8, 1),
    (masks.config_strided(16, 2, 4), 8, 1),                      # 256 lines
    (masks.config_causal(17), 8, 1),                             # 272
    (masks.config_global_local(16), 16, 1),                      # 512
    (masks.config_strided(17, 2, 4), 8, 2),                      # 544
])
def test_one_launch_equals_two(lib, mask, nh, batch):
    g = torch.Generator(device=DEV).manual_seed(nh)
    mk = lambda n: torch.randn(batch, n * 128, nh, 128, device=DEV, generator=g).to(torch.bfloat16)
    q, k, v, do = mk(mask.shape[0]), mk(mask.shape[1]), mk(mask.shape[1]), mk(mask.shape[0])
    tl = build_tile_list(mask, 128)
    d = tl.on(DEV)
    o, lse = ops.bsa_fwd(q, k, v, tl, SCALE)
    delta = ops.softmax_delta(o, do)
    got = ops.bsa_bwd(do, q, k, v, None, lse, tl, SCALE, softmax_d=delta)
    dq, dk, dv = (torch.full_like(t, 7.0) for t in (q, k, v))
    s3, st = _lib.strides3, torch.cuda.current_stream().cuda_stream
    ins = [t.data_ptr() for t in (q, k, v, do, lse, delta)]
    size = (batch, nh, tl.n_qtiles, tl.n_ktiles, tl.nnz, 128)
    lists = lambda *n: [d[x].data_ptr() for x in n]
    assert lib.ua_bsa_bwd_dkdv(*ins, dk.data_ptr(), dv.data_ptr(), *lists("col_ptr", "row_idx", "cflag", "k_order"), *size,
                               s3(q), s3(k), s3(v), s3(do), s3(dk), s3(dv), SCALE, st) == 0
    assert lib.ua_bsa_bwd_dq(*ins, dq.data_ptr(), *lists("row_ptr", "col_idx", "flag", "q_order"), *size,
                             s3(q), s3(k), s3(v), s3(do), s3(dq), SCALE, st) == 0
    torch.cuda.synchronize()
    for a, b in zip(got, (dq, dk, dv)):
        assert torch.equal(a, b)
