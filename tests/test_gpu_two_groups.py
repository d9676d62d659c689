"""Workgroups of one, two and four groups per tile line: walks of no tile, one tile and an odd number of them, rows whose
causal tile is not the last one (tile lists, one group), and dense launches on both sides of every bound at which the
groups are chosen."""
import numpy as np
import pytest
import torch

from oracle import attn_oracle as ao
from tests.gpu_util import ATOL_O, RTOL_LSE, SCALE, lse_rel_err, max_abs
from ultraattn_amd import ops
from ultraattn_amd.flash_attn_interface import _flash_attn_backward, _flash_attn_forward

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(sq, sk, nh, seed=5):
    g = torch.Generator().manual_seed(seed)
    mk = lambda n: torch.randn(1, n, nh, 128, generator=g).to(torch.bfloat16)
    return mk(sq), mk(sk), mk(sk), mk(sq)


def _check(got, q, k, v, do, keep, heads):
    o, lse, dq, dk, dv = got
    for h in heads:
        s = slice(h, h + 1)
        cut = [t[:, :, s] for t in (q, k, v, do)]
        ro, rl = ao.dense_fwd(*cut[:3], SCALE, keep)
        rq, rk, rv = ao.dense_bwd_autograd(*cut, SCALE, keep)
        assert max_abs(o[:, :, s], ro) <= ATOL_O and lse_rel_err(lse[:, s], rl) <= RTOL_LSE
        for a, b in ((dq, rq), (dk, rk), (dv, rv)):
            assert max_abs(a[:, :, s], b) <= 2e-2


@pytest.mark.parametrize("mask", [
    [[2]], [[0, 0], [1, 0]], [[2, 1, 1]], [[1, 2, 1], [2, 0, 0], [0, 0, 2]], [[1, 1, 1, 1, 1]],
])
def test_short_and_odd_walks(mask):
    mask = np.array(mask, np.uint8)
    q, k, v, do = _inputs(mask.shape[0] * 128, mask.shape[1] * 128, 3)
    d = [t.to(DEV) for t in (q, k, v, do)]
    o, lse = ops.bsa_fwd(*d[:3], mask, SCALE, block=128)
    g = ops.bsa_bwd(d[3], *d[:3], o, lse, mask, SCALE, block=128)
    _check((o, lse, *g), q, k, v, do, ao.element_mask(mask, 128), range(3))


@pytest.mark.parametrize("sq,sk,nh,causal", [
    (512, 128, 2, True),                                         # rows above the first key: empty walks
    (128, 128, 128, False), (128, 128, 129, True),               # backward: 256 and 258 lines
    (256, 256, 32, False), (256, 384, 27, False),                # 128 and 135: four groups and two
    (1024, 1024, 16, True), (2048, 2048, 8, True),               # causal, 256 in the backward, four groups
    (256, 2048, 2, True),                                        # cut rows with four groups
    (128, 256, 256, True), (384, 128, 86, False),                # forward: 256 and 258
    (2048, 2048, 16, True), (2048, 2048, 17, True),              # causal, long walks: 512 and 544 in the backward
    (2176, 1920, 9, True),                                       # 153 rows, 135 columns, bottom-right aligned
    (128, 384, 100, False), (128, 384, 150, False),              # walks of three: four groups and two
    (640, 384, 20, True),                                        # four groups, walks of none to three
    (1920, 1920, 17, True),                                      # two groups, walks of one to fifteen
])
def test_around_the_bounds(sq, sk, nh, causal):
    q, k, v, do = _inputs(sq, sk, nh)
    d = [t.to(DEV) for t in (q, k, v, do)]
    r = _flash_attn_forward(*d[:3], 0.0, SCALE, causal)
    g = _flash_attn_backward(d[3], *d[:3], r[0], r[5], None, None, None, 0.0, SCALE, causal)
    keep = torch.ones(sq, sk, dtype=torch.bool)
    if causal:
        keep = torch.arange(sk)[None, :] <= torch.arange(sq)[:, None] + (sk - sq)
    _check((r[0], r[5], *g[:3]), q, k, v, do, keep, (0, nh - 1))


@pytest.mark.parametrize("sq,sk,nh,causal", [
    (128, 128, 65, False), (128, 128, 128, True),                # half lines: 130 and 256 lines of one tile
    (512, 512, 32, True), (128, 256, 85, True),                  # 256 and 255 lines
    (1024, 1024, 12, True), (1024, 1024, 13, True),              # 192 and 208 uneven ones: four groups, half lines
    (1536, 1536, 10, True),                                      # 240 that average six tiles: four groups
    (512, 512, 40, True), (512, 512, 41, True),                  # 320 and 328
    (512, 512, 48, True), (512, 512, 49, True),                  # 384 and 392 that average four tiles
    (640, 640, 51, True), (640, 640, 52, True),                  # 510 and 520 that average five
    (512, 640, 35, True), (512, 640, 36, True),                  # 315 and 324 with more keys than queries
    (384, 384, 50, True), (256, 256, 65, True),                  # 300 of three tiles at most; 260 of two: one group
    (128, 128, 130, True), (256, 256, 70, True),                 # 260 of one tile, 280 of one or two
    (512, 128, 50, True), (128, 640, 42, False),                 # empty walks on half lines; odd walks of one and five
    (128, 256, 43, False), (256, 128, 44, True),                 # 86 and 43, 44 and 88 lines a side: the last 8 of a side not full
    (384, 384, 23, False), (256, 256, 33, True), (128, 384, 33, True),      # halves of 69, of 66, of 33 and 99
    (2048, 256, 6, False), (640, 1408, 5, False),                # cut columns on half lines; odd walks of five and eleven
    (384, 2560, 4, False), (256, 2816, 4, True),                 # cut rows on half lines
])
def test_half_lines(sq, sk, nh, causal):
    test_around_the_bounds(sq, sk, nh, causal)


@pytest.mark.parametrize("sq,sk,nh", [(512, 512, 64), (512, 512, 65), (384, 640, 96), (512, 384, 90), (128, 128, 256)])
def test_two_to_three_workgroups_per_cu(sq, sk, nh):
    """512 and 520 lines, 768 with longer rows, 630 with longer columns, 512 of one tile: where the rows' wavefronts go first and where not."""
    test_around_the_bounds(sq, sk, nh, False)


@pytest.mark.parametrize("sq,sk,nh", [
    (896, 512, 12), (768, 640, 1), (896, 768, 1), (896, 896, 1),         # four groups of 132 lines; cuts of both sides in halves, of columns and of both in four
    (128, 768, 1), (128, 1536, 20), (128, 1536, 40),                     # rows cut in halves: 7, 260 and 520 lines
    (128, 2048, 6), (128, 2688, 24), (256, 2688, 32),                    # rows cut, one group: 102, 528 and 736
    (1536, 128, 20), (128, 1280, 48), (512, 128, 48),                    # whole lines: 260 and 528 in halves, 240 short ones of one group
    (640, 256, 109), (640, 256, 110), (512, 2048, 40),                   # 763 and 770, on both sides of the last bound; 800 with cut rows
])
def test_causal_plans(sq, sk, nh):
    """Every form with every kind of cut that a causal backward takes."""
    test_around_the_bounds(sq, sk, nh, True)
