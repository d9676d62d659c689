"""Workspaces of cut dense calls: none is kept for calls that are not cut, and threads that share a stream share one
without mixing their partial results."""
import threading

import pytest
import torch

from tests.gpu_util import ATOL_O, SCALE
from ultraattn_amd import flash_attn_interface as fai
from ultraattn_amd.flash_attn_interface import _flash_attn_backward, _flash_attn_forward

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(sq, sk, nh, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    mk = lambda n: torch.randn(1, n, nh, 128, device=DEV, generator=g).to(torch.bfloat16)
    return mk(sq), mk(sk), mk(sk), mk(sq)


def _pass(q, k, v, do, causal):
    r = _flash_attn_forward(q, k, v, 0.0, SCALE, causal)
    return (r[0], r[5]) + _flash_attn_backward(do, q, k, v, r[0], r[5], None, None, None, 0.0, SCALE, causal)


def test_calls_that_are_not_cut_keep_nothing(lib):
    fai._workspaces.clear()
    for sq, sk, nh, causal in ((512, 512, 32, False), (1024, 1024, 8, False), (2304, 3456, 32, True)):
        _pass(*_inputs(sq, sk, nh, 0), causal)
    assert not fai._workspaces
    # an output that is not contiguous is not cut either
    q, k, v, _ = _inputs(1024, 4096, 1, 0)
    _flash_attn_forward(q, k, v, 0.0, SCALE, False, out=torch.empty(1, 1024, 2, 128, dtype=torch.bfloat16, device=DEV)[:, :, :1])
    assert not fai._workspaces
    _flash_attn_forward(q, k, v, 0.0, SCALE, False)
    assert [t.numel() for t in fai._workspaces.values()] == [lib.ua_dense_workspace_used(1, 1, 1024, 4096, 0, 0)]


@pytest.mark.parametrize("n_threads,own_streams", [(4, False), (4, True)])
def test_threads(n_threads, own_streams):
    """Each thread repeats its own forward and backward, both cut; on one stream all of them use the same workspace."""
    shapes = [(1024, 4096, 1, False), (256, 2048, 2, True), (512, 4096, 1, False), (1024, 4096, 1, True)][:n_threads]
    ins = [_inputs(*s[:3], seed=i) for i, s in enumerate(shapes)]
    want = [_pass(*x, s[3]) for x, s in zip(ins, shapes)]
    torch.cuda.synchronize()
    wrong, start = [], threading.Barrier(n_threads)

    def work(i):
        stream = torch.cuda.Stream() if own_streams else torch.cuda.current_stream()
        start.wait()
        with torch.cuda.stream(stream):
            for rep in range(50):
                got = _pass(*ins[i], shapes[i][3])
                if rep % 10 == 9:
                    stream.synchronize()
                    wrong.extend((i, rep, j) for j, (a, b) in enumerate(zip(got, want[i])) if not torch.equal(a, b))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(n_threads)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong


@pytest.mark.parametrize("nh", [255, 256, 257])
def test_heads_beyond_the_merge(nh):
    """A forward of few lines and many heads with a long walk: the merge of a cut takes 256 heads, more run uncut."""
    sq, sk = 128, 8192
    q, k, v, _ = _inputs(sq, sk, nh, 1)
    r = _flash_attn_forward(q, k, v, 0.0, SCALE, False)
    for h in (0, nh - 1):
        s = (q[0, :, h].float() @ k[0, :, h].float().T) * SCALE
        assert (r[0][0, :, h].float() - torch.softmax(s, -1) @ v[0, :, h].float()).abs().max().item() <= ATOL_O
        assert (r[5][0, h] - torch.logsumexp(s, -1)).abs().max().item() <= 1e-4
