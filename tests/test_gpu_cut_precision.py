"""A dense forward that has room to be cut is as exact as the same rectangle walked whole, where a cut would only save a little time: the
partial results of a cut are bf16, and their rounding adds a fifth to the error of a result that is cut in two."""
import pytest
import torch

from tests.gpu_util import SCALE
from tests.test_gpu_dense import dense_unsplit
from ultraattn_amd.flash_attn_interface import _flash_attn_forward

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("nh,seq", [(8, 4480), (5, 8192), (3, 4480)])
def test_error_is_that_of_whole_walks(lib, nh, seq):
    g = torch.Generator(device=DEV).manual_seed(seq)
    q, k, v = (torch.randn(1, seq, nh, 128, device=DEV, generator=g).to(torch.bfloat16) for _ in range(3))
    got = _flash_attn_forward(q, k, v, 0.0, SCALE, False)[0]
    whole = dense_unsplit(lib, q, k, v, q, False)[0]
    for h in (0, nh - 1):
        p = torch.softmax((q[0, :, h].double() @ k[0, :, h].double().T) * SCALE, -1)
        want = p @ v[0, :, h].double()
        err, err_whole = ((x[0, :, h].double() - want).norm().item() for x in (got, whole))
        assert err <= 1.02 * err_whole, (h, err / err_whole)           # the mean over half a million values and more is good to 1 %


def test_rectangles_that_stay_whole(lib):
    """As above, and more of the kind (host arithmetic)."""
    for nh, seqs in ((8, range(4224, 4993, 128)), (5, range(7808, 9473, 128)), (3, (4480, 5248))):
        for s in seqs:
            assert lib.ua_dense_workspace_used(1, nh, s, s, 0, 0) == 0, (nh, s)


@pytest.mark.gpu
@pytest.mark.parametrize("nh,sq,sk", [(10, 1664, 6656), (24, 768, 2944), (28, 1152, 4096), (48, 768, 2944), (43, 384, 2048), (65, 256, 2048), (9, 2432, 4608)])
def test_causal_rectangles_in_two_rounds_are_cut_and_rounded_once(lib, nh, sq, sk):
    """Long causal lines: 130, 144 and 252 in four groups, 288 in two; then 129 and 130 short ones, and 171 whose last part the first
    rows do not reach."""
    g = torch.Generator(device=DEV).manual_seed(sk)
    q, k, v = (torch.randn(1, n, nh, 128, device=DEV, generator=g).to(torch.bfloat16) for n in (sq, sk, sk))
    rows = nh * sq
    assert lib.ua_dense_workspace_used(1, nh, sq, sk, 1, 0) >= 2 * rows * (128 * 4 + 4)          # two parts or more, fp32
    assert lib.ua_dense_workspace_bytes(1, nh, sq, sk, 0) >= lib.ua_dense_workspace_used(1, nh, sq, sk, 1, 0)
    got = _flash_attn_forward(q, k, v, 0.0, SCALE, True)
    whole = dense_unsplit(lib, q, k, v, q, True)
    hidden = torch.ones(sq, sk, dtype=torch.bool, device=DEV).triu(sk - sq + 1)
    for h in (0, nh - 1):
        s = ((q[0, :, h].double() @ k[0, :, h].double().T) * SCALE).masked_fill(hidden, -torch.inf)
        want, lse = torch.softmax(s, -1) @ v[0, :, h].double(), torch.logsumexp(s, -1)
        err, err_whole = ((x[0][0, :, h].double() - want).norm().item() for x in (got, whole))
        assert err <= 1.02 * err_whole, (h, err / err_whole)
        assert ((lse_of(got)[0, h] - lse).abs() / lse.abs()).max().item() <= 1e-5


def lse_of(result):
    return next(x for x in result if torch.is_tensor(x) and x.dtype == torch.float32 and x.dim() == 3)
