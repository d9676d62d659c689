"""delta at every number of tokens per workgroup, with sequences that do not fill the last one."""
import pytest
import torch

from ultraattn_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,S,nh", [(1, 5, 32), (1, 2051, 32), (2, 2049, 17), (1, 9001, 32), (1, 16390, 3), (1, 65539, 1), (3, 33, 200)])
def test_delta_sizes(B, S, nh):
    g = torch.Generator(device=DEV).manual_seed(S)
    o, do = (torch.randn(B, S, nh, 128, device=DEV, generator=g).to(torch.bfloat16) for _ in range(2))
    ref = (o.double() * do.double()).sum(-1).transpose(1, 2)
    assert (ops.softmax_delta(o, do).double() - ref).abs().max().item() <= 1e-4
