"""Dense forwards whose last lines run as a cut rectangle of their own: one and two sequences, one to a quarter of a wave left
over, parts that do not divide the keys.  Against the same call without a workspace (one launch, no cut), and against
fp64: the rows of the cut lines are as exact as those of the whole ones."""
import pytest
import torch

from tests.gpu_util import SCALE, lse_rel_err
from ultraattn_amd import _lib
from ultraattn_amd.flash_attn_interface import _flash_attn_forward

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("B,nh,sq,sk", [
    (1, 32, 2304, 3456), (2, 16, 2176, 3456), (1, 3, 21888, 2560), (1, 32, 2560, 4096), (1, 5, 13312, 3328),
])
def test_tail_equals_the_single_launch(lib, B, nh, sq, sk):
    assert lib.ua_dense_workspace_bytes(B, nh, sq, sk, 0) > 0
    g = torch.Generator(device=DEV).manual_seed(sq)
    mk = lambda n: torch.randn(B, n, nh, 128, device=DEV, generator=g).to(torch.bfloat16)
    q, k, v = mk(sq), mk(sk), mk(sk)
    res = _flash_attn_forward(q, k, v, 0.0, SCALE, False)
    o, lse = torch.full_like(q, 7.0), torch.full((B, nh, sq), 7.0, device=DEV)
    s3 = _lib.strides3
    assert lib.ua_dense_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), B, nh, sq, sk, 128, s3(q), s3(k), s3(v), s3(o),
                            SCALE, 0, None, 0, torch.cuda.current_stream().cuda_stream) == 0
    # Both round the result once (to a bf16 step, 2^-7 of the value) and the P of a key once, against references that differ
    # between parts: sqrt(2) 2^-9 / sqrt(3) of an output's standard deviation, 0.033 on average and up to 0.066 in the rows
    # whose weights concentrate on few keys: 1e-4, of which the largest of ten million may be six.  (No error at all is
    # bounded by 2^-8 sum(p |v|) = 3e-3; wrong weights of the parts give up to 1e-2.)
    d = (res[0].float() - o.float()).abs()
    worst = (d - 2 ** -7 * o.float().abs()).max().item()
    assert worst <= 6e-4 and lse_rel_err(res[5], lse.cpu()) <= 1e-5
    # every row against fp64.  The keys of a row are 20 tiles and more of N(0, 1), so all rows have the same error, from the
    # rounding of P and of the result; a further rounding of the parts would add to it in the cut rows (by 20 %), wrong
    # weights of the parts far more.  The mean over 16384 values and more is good to 2 %.
    tiles = sq // 128
    whole = (512 * (B * nh * tiles // 512)) // (B * nh)         # query tiles of a sequence that run in full waves
    cut = slice(128 * whole, sq)
    for b, h in {(0, 0), (B - 1, nh - 1)}:
        s = (q[b, :, h].double() @ k[b, :, h].double().T) * SCALE
        want = torch.softmax(s, -1) @ v[b, :, h].double()
        err, err_cut = _rel(res[0][b, :128 * whole, h], want[:128 * whole]), _rel(res[0][b, cut, h], want[cut])
        assert err <= 5e-3 and err_cut <= 1.05 * err, (err, err_cut)
        assert lse_rel_err(res[5][b, h, cut], torch.logsumexp(s, -1)[cut].float().cpu()) <= 1e-5


@pytest.mark.parametrize("key", [0, 3455])
def test_infinities_stay_where_they_belong(lib, key):
    """An infinite value of the first or the last part (seven here) reaches the outputs it belongs to, cut lines and whole ones
    alike, and turns none into NaN."""
    nh, sq, sk = 32, 2304, 3456
    g = torch.Generator(device=DEV).manual_seed(key)
    mk = lambda n: torch.randn(1, n, nh, 128, device=DEV, generator=g).to(torch.bfloat16)
    q, k, v = mk(sq), mk(sk), mk(sk)
    v[0, key, :, 5] = float("inf")
    v[0, key, :, 6] = float("-inf")
    o = _flash_attn_forward(q, k, v, 0.0, SCALE, False)[0].float()
    assert (o[..., 5] == float("inf")).all() and (o[..., 6] == float("-inf")).all()
    assert torch.isfinite(o[..., :5]).all() and torch.isfinite(o[..., 7:]).all()
