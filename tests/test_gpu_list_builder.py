"""The device builder where its ranking can go wrong (identical lists, lists that first differ around one
comparison round of 256 indices, more lines than one round of keys, a last workgroup that is not full),
and masks handed over with the call on both sides of the host / device choice."""
import numpy as np
import pytest
import torch

from oracle import tilelist_oracle as to
from tests.gpu_util import SCALE, seeded_inputs
from ultraattn_amd import masks, ops
from ultraattn_amd.tilelist import build_tile_list, build_tile_list_device

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FIELDS = ("row_ptr", "col_idx", "flag", "col_ptr", "row_idx", "cflag", "q_order", "k_order")


def _late_differences(n_rows, n_cols):
    m = np.ones((n_rows, n_cols), np.uint8)
    for r in range(n_rows):                     # one hole per row, around index 256 of the list
        m[r, (253 + r) % n_cols] = 0
    return m


@pytest.mark.parametrize("make,block", [
    (lambda: np.ones((9, 300), np.uint8), 128), (lambda: np.ones((2, 1), np.uint8), 128), (lambda: np.full((1, 1), 2, np.uint8), 384),
    (lambda: _late_differences(8, 300), 128), (lambda: _late_differences(8, 300).T.copy(), 128),
    (lambda: np.tril(np.full((70, 70), 1, np.uint8)) + np.eye(70, dtype=np.uint8), 512),
    (lambda: masks.config_strided(300), 512), (lambda: np.random.RandomState(8).randint(0, 3, size=(1030, 3)).astype(np.uint8), 128),
])
def test_device_lists(make, block):
    m = make()
    want = to.build_tile_list(m, block // 128)
    got = build_tile_list_device(torch.from_numpy(m).to(DEV), block, nnz=want["col_idx"].shape[0])
    for f in FIELDS:
        assert np.array_equal(got[f].cpu().numpy(), want[f]), f


@pytest.mark.parametrize("n,block", [(4, 128), (16, 512), (20, 512)])
def test_mask_with_the_call_equals_kept_plan(n, block):
    for mask in (masks.config_causal(n), np.ones((n, n), np.uint8)):      # 4096 tiles and less: built on the host
        q, k, v, do = (t.to(DEV) for t in seeded_inputs(mask, block, 3, nh=1))
        tl = build_tile_list(mask, block)
        a, b = ops.bsa_fwd(q, k, v, mask, SCALE, block=block), ops.bsa_fwd(q, k, v, tl, SCALE)
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
        ga = ops.bsa_bwd(do, q, k, v, *a, mask, SCALE, block=block)
        gb = ops.bsa_bwd(do, q, k, v, *b, tl, SCALE)
        assert all(torch.equal(x, y) for x, y in zip(ga, gb))
