"""The device builder's two launches against the host builder at the edges of what they take (256 blocks a side, 64 tiles a block)
and where two lines' keys are equal and their blocks decide: read from either end, over rows and columns, at the borders of the words that hold the blocks' bits, with
CAUSAL blocks where the lines part, and one list ending inside the other."""
import numpy as np
import pytest
import torch

from ultraattn_amd import _lib
from ultraattn_amd.tilelist import build_tile_list, build_tile_list_device

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FIELDS = ("row_ptr", "col_idx", "flag", "col_ptr", "row_idx", "cflag", "q_order", "k_order")


def _check(m, rate):
    m = np.ascontiguousarray(m.astype(np.uint8))
    want = build_tile_list(m, 128 * rate)
    got = build_tile_list_device(torch.from_numpy(m).to(DEV), 128 * rate, nnz=want.nnz, check=True)
    for f in FIELDS:
        w = getattr(want, f)
        assert np.array_equal(got[f].cpu().numpy()[:w.shape[0]], w), (m.shape, rate, f)


@pytest.mark.parametrize("shape,rate", [((256, 256), 1), ((257, 3), 2), ((3, 257), 2), ((256, 2), 16), ((5, 4), 64), ((5, 4), 65), ((1, 256), 3), ((33, 31), 7)])
def test_edges_of_the_range(shape, rate):
    rs = np.random.RandomState(shape[0] + rate)
    _check(rs.randint(0, 3, size=shape), rate)
    _check((rs.rand(*shape) < 0.03) * rs.randint(1, 3, size=shape), rate)          # empty lines among them


@pytest.mark.parametrize("at", [0, 1, 31, 32, 63, 64, 127, 128, 191, 192, 254, 255])
@pytest.mark.parametrize("rate", [1, 4])
def test_lines_that_part_at_one_block(at, rate):
    rs = np.random.RandomState(at)
    m = np.tile(rs.randint(0, 3, size=256), (12, 1))
    m[:, 0] = m[:, 255] = 1                                  # the same ends, from either side
    for r in range(12):
        m[r, at] = r % 3                                     # EMPTY, FULL, CAUSAL
    m[8:, (at + 1) % 256] = 0                                # of equal length again
    for flip in (m, m[:, ::-1]):
        _check(flip, rate)
        _check(flip.T, rate)


@pytest.mark.parametrize("rate", [2, 3, 5])
def test_few_different_lines(rate):
    rs = np.random.RandomState(rate)
    for n, k in ((64, 65), (130, 100), (200, 256)):
        base = rs.randint(0, 3, size=(3, k))
        m = base[rs.randint(0, 3, size=n)].copy()
        for _ in range(n // 2):
            m[rs.randint(n), rs.randint(k)] = rs.randint(3)
        _check(m, rate)
        _check(m.T, rate)


def test_scratch_that_does_not_fit_leaves_the_lists_the_same(lib):
    m = torch.from_numpy(np.random.RandomState(1).randint(0, 3, size=(20, 30)).astype(np.uint8)).to(DEV)
    want = build_tile_list(m.cpu().numpy(), 256)
    need = lib.ua_tilelist_scratch_bytes(20, 30, 2)
    assert need > 0 and lib.ua_tilelist_scratch_bytes(257, 30, 2) == lib.ua_tilelist_scratch_bytes(20, 30, 65) == 0
    space = torch.empty(need + 32, dtype=torch.uint8, device=DEV)
    base = (space.data_ptr() + 15) // 16 * 16
    for scratch, size in ((None, 0), (base, need - 1), (base + 8, need), (base, need)):
        out = {f: torch.full((max(4, getattr(want, f).shape[0]),), 77, dtype=torch.uint8 if "flag" in f else torch.int32, device=DEV) for f in FIELDS}
        work = torch.full((107,), -1, dtype=torch.int32, device=DEV)
        rc = lib.ua_tilelist_build_device_scratch(m.data_ptr(), 20, 30, 2, *(out[f].data_ptr() for f in FIELDS), work.data_ptr(), scratch, size,
                                                  torch.cuda.current_stream().cuda_stream)
        assert rc == 0, lib.ua_strerror(rc)
        torch.cuda.synchronize()
        assert int(work[102]) == 0
        for f in FIELDS:
            w = getattr(want, f)
            assert np.array_equal(out[f].cpu().numpy()[:w.shape[0]], w), (scratch, size, f)


@pytest.mark.parametrize("rows,cols,rate", [(1, 1, 1), (3, 5, 2), (16, 16, 4), (33, 31, 4), (257, 255, 1), (1031, 1031, 1)])
def test_lists_of_a_mask_on_the_host(rows, cols, rate):
    """Copied over as lists or as a mask, of sizes that are no multiple of 16 bytes, the largest beyond 1 MiB."""
    from ultraattn_amd._lib import native
    m = np.random.RandomState(rows).randint(0, 3, size=(rows, cols)).astype(np.uint8)
    if rows > 1000:
        m *= np.random.RandomState(1).rand(rows, cols) < 0.05
    want = build_tile_list(m, 128 * rate)
    buf, nqt, nkt, nnz = native().lists_from_mask(m, rows, cols, rate, 0)
    assert (nqt, nkt, nnz) == (rows * rate, cols * rate, want.nnz)
    got, at = buf.cpu().numpy(), 0
    for f in ("row_ptr", "col_ptr", "q_order", "k_order", "col_idx", "row_idx"):
        w = getattr(want, f)
        assert np.array_equal(got[at:at + len(w)], w), f
        at += len(w)
    for f in ("flag", "cflag"):
        w = getattr(want, f)
        assert np.array_equal(got[at:at + (nnz + 3) // 4].view(np.uint8)[:nnz], w[:nnz]), f
        at += (nnz + 3) // 4
