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


def _emulated(q, k, v, groups, alone):
    """O of one head in fp64, P rounded to bf16, by the kernels' schedule: each group of waves walks the keys 128 / groups (at most 64) at
    a time; a row sum of 2^24 or more raises the reference max of that row `alone` or of the 32 rows of its wave."""
    q, k, v = (t[0, :, 0].double().cpu() for t in (q, k, v))
    s = (q @ k.t().contiguous()) * (SCALE * 1.4426950408889634)
    step, parts = min(64, 128 // groups), []
    for g in range(groups):
        starts = [t + step * g for t in range(0, k.shape[0], 128)] if groups > 1 else range(0, k.shape[0], step)
        m = None
        for at in starts:
            x, w = s[:, at:at + step], v[at:at + step]
            if m is None:
                m, l, o = x.amax(1), torch.zeros(len(x), dtype=torch.float64), torch.zeros(len(x), 128, dtype=torch.float64)
            else:
                over = torch.exp2(x - m[:, None]).sum(1) >= 2.0 ** 24
                if not alone:
                    over = over.view(-1, 32).any(1).repeat_interleave(32)
                new = torch.where(over, torch.maximum(m, x.amax(1)), m)
                l, o, m = l * torch.exp2(m - new), o * torch.exp2(m - new)[:, None], new
            p = torch.exp2(x - m[:, None])
            l, o = l + p.sum(1), o + p.to(torch.bfloat16).double() @ w
        parts.append((m, l, o))
    top = torch.stack([m for m, _, _ in parts]).amax(0)
    weights = [torch.exp2(m - top) for m, _, _ in parts]
    total = sum(w * l for w, (_, l, _) in zip(weights, parts))
    return (sum(w[:, None] * o for w, (_, _, o) in zip(weights, parts)) / total[:, None]).to(torch.bfloat16)


@pytest.mark.parametrize("heads,groups", [(1, 4), (128, 1)])
def test_the_rows_of_a_wave_raise_their_reference_together(heads, groups):
    """Every third row's scores outgrow the reference in the walk, the others' do not but are rescaled with them: O is that of this schedule
    (but for entries within fp32 rounding of the middle between two bf16), not that of rows that are raised alone."""
    g = torch.Generator().manual_seed(3)
    q, k, v = _rows(512, heads, g), _rows(512, heads, g), _rows(512, heads, g)
    k = (k.float() * torch.logspace(-1, 1, 512, device=DEV).view(1, -1, 1, 1)).to(torch.bfloat16)
    q = (q.float() * torch.where(torch.arange(512, device=DEV) % 3 == 0, 1.0, 0.02).view(1, -1, 1, 1)).to(torch.bfloat16)
    o = _flash_attn_forward(q, k, v, 0.0, SCALE, False)[0]
    for h in (0, heads - 1):
        cut = [t[:, :, h:h + 1] for t in (q, k, v)]
        together, alone = (int((o[0, :, h].cpu() != _emulated(*cut, groups, x)).sum()) for x in (False, True))
        assert together < alone / 2, (together, alone)
