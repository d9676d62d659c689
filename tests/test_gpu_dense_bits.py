"""What the bits of a dense forward depend on.  The flash-attention signatures return delta = rowsum(dO * O) in fp32, in which a
row whose sums are taken in another order shows at once."""
import pytest
import torch

from tests.gpu_util import SCALE
from ultraattn_amd.flash_attn_interface import _flash_attn_backward, _flash_attn_forward

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rows(tokens, heads, g):
    return torch.randn(1, tokens, heads, 128, generator=g).to(torch.bfloat16).to(DEV)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("sq,few,many", [(128, 1, 129), (128, 64, 250), (512, 8, 70)])
def test_one_key_tile_is_walked_by_one_group(sq, few, many, causal):
    """Rows that meet a single tile of keys: the same bits beside up to 128 lines and beside more."""
    g = torch.Generator().manual_seed(sq + few)
    q, k, v, do = _rows(sq, many, g), _rows(128, many, g), _rows(128, many, g), _rows(sq, many, g)

    def outputs(heads):
        x = [t[:, :, :heads] for t in (q, k, v, do)]
        o, lse = [_flash_attn_forward(*x[:3], 0.0, SCALE, causal)[i] for i in (0, 5)]
        return o, lse, _flash_attn_backward(x[3], *x[:3], o, lse, None, None, None, 0.0, SCALE, causal)[3]

    (o, lse, delta), (many_o, many_lse, many_delta) = outputs(few), outputs(many)
    assert torch.equal(o, many_o[:, :, :few]) and torch.equal(lse, many_lse[:, :few]) and torch.equal(delta, many_delta[:, :few])
