"""Tile lists of few lines, which run with eight waves a workgroup: bit for bit what the same heads give in a launch of many
lines, also where rows raise their reference max in the middle of the walk, and against the oracle."""
import numpy as np
import pytest
import torch

from oracle import attn_oracle as ao
from tests.gpu_util import ATOL_O, RTOL_LSE, SCALE, lse_rel_err, max_abs
from ultraattn_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _mask(kind, n):
    if kind == "random":
        m = np.random.default_rng(n).integers(0, 3, (n, n)).astype(np.uint8)
        m[n // 2] = 0                                                    # rows without keys
        return m
    return np.tril(np.ones((n, n), np.uint8), -1) + 2 * np.eye(n, dtype=np.uint8) if kind == "causal" else np.ones((n, n), np.uint8)


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("kind,blocks,heads", [
    ("causal", 1, 1), ("causal", 2, 3), ("causal", 64, 4),               # one line, a few, 256
    ("full", 1, 2), ("full", 16, 8), ("full", 43, 3),                    # 128, and 129 of full length (four waves)
    ("random", 5, 1), ("random", 66, 2),                                 # walks of more than 64 entries
])
def test_same_bits_as_a_long_launch(kind, blocks, heads, grow):
    mask, n = _mask(kind, blocks), blocks * 128
    g = torch.Generator().manual_seed(blocks)
    q, k, v = (torch.randn(1, n, heads, 128, generator=g) for _ in range(3))
    if grow:
        k = k * torch.logspace(-1, 1, n).view(1, -1, 1, 1)
        q = q * torch.where(torch.arange(n) // 16 % 2 == 0, 1.0, 0.02).view(1, -1, 1, 1)
    few = [t.to(torch.bfloat16).to(DEV) for t in (q, k, v)]
    many = [t.repeat(1, 1, 512 // (blocks * heads) + 1, 1) for t in few]
    o, lse = ops.bsa_fwd(*few, mask, SCALE, block=128)
    long_o, long_lse = ops.bsa_fwd(*many, mask, SCALE, block=128)
    assert torch.equal(o, long_o[:, :, :heads]) and torch.equal(lse, long_lse[:, :heads])
    if not grow and blocks <= 16:
        ro, rl = ao.dense_fwd(*[t[:, :, :1].to(torch.bfloat16) for t in (q, k, v)], SCALE, ao.element_mask(mask, 128))
        assert max_abs(o[:, :, :1], ro) <= ATOL_O and lse_rel_err(lse[:, :1], rl) <= RTOL_LSE
