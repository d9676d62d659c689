"""Dense forwards whose last lines run as a cut rectangle of their own, against the same call without a workspace (one
launch, no cut): one and two sequences, one to a quarter of a wave left over, parts that do not divide the keys."""
import pytest
import torch

from tests.gpu_util import SCALE, lse_rel_err, max_abs
from ultraattn_amd import _lib
from ultraattn_amd.flash_attn_interface import _flash_attn_forward

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


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
    assert max_abs(res[0], o.cpu()) <= 8e-3 and lse_rel_err(res[5], lse.cpu()) <= 1e-5
