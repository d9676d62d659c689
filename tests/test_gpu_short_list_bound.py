"""Full lists on both sides of the number of lines up to which they run with eight waves a workgroup: the same bits as in a launch of many lines."""
import numpy as np
import pytest
import torch

from tests.gpu_util import SCALE
from ultraattn_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("blocks,heads", [(32, 7), (25, 9), (17, 15), (16, 16), (4, 64), (3, 86)])      # 224, 225 and 255 long lines; 256, 256 and 258 of up to 16 tiles
def test_same_bits_around_the_bound(blocks, heads):
    g = torch.Generator().manual_seed(heads)
    few = [torch.randn(1, blocks * 128, heads, 128, generator=g).to(torch.bfloat16).to(DEV) for _ in range(3)]
    many = [t.repeat(1, 1, 3, 1) for t in few]
    mask = np.ones((blocks, blocks), np.uint8)
    o, lse = ops.bsa_fwd(*few, mask, SCALE, block=128)
    many_o, many_lse = ops.bsa_fwd(*many, mask, SCALE, block=128)
    assert torch.equal(o, many_o[:, :, :heads]) and torch.equal(lse, many_lse[:, :heads])
