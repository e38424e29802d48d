"""qvex_gdn_conv_qk on prompt chunks (8 consecutive tokens per wave from 1024 blocks
of 512 channels on, below that a token per wave) against the same tokens in calls
of 8 or fewer: the same bits in q, k, v, a, b and in the ring, at partial runs, ring
wrap-around and every position of the state rows."""

import pytest
import torch

from qvex import _C
from qvex.kernels import _ptr, _stream

DEV = "cuda:0"


def conv(proj, ring, pos, cw, C, key_dim, Hv, ab_off):
    T = proj.shape[0]
    out = [torch.zeros((T, n), dtype=torch.bfloat16, device=DEV) for n in (key_dim, key_dim, C - 2 * key_dim, Hv, Hv)]
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    _C.call("qvex_gdn_conv_qk", _ptr(proj), proj.stride(0), _ptr(ring), ring.shape[0], _ptr(p), _ptr(cw), cw.shape[1],
            *[_ptr(t) for t in out], T, C, key_dim, Hv, ab_off, 0.0078, 0.088, 1e-6, _stream())
    torch.cuda.synchronize()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("T,pos,spare", [(9, 0, 0), (15, 2, 1), (16, 1000, 0), (17, 14, 5), (40, 39, 0), (131, 7, 64)])
@pytest.mark.parametrize("C,key_dim,Hv", [(1024, 256, 4), (1536, 128, 40)])
def test_conv_runs_match_single_tokens(T, pos, spare, C, key_dim, Hv):
    check(T, pos, spare, C, key_dim, Hv)


@pytest.mark.gpu
@pytest.mark.parametrize("T,pos,spare", [(64, 5, 0), (65, 0, 0), (66, 68, 1), (71, 1000, 0), (72, 74, 5), (131, 7, 64)])
def test_conv_runs_of_8_tokens_match_single_tokens(T, pos, spare):
    """64 tokens of 8192 channels are the last call with a token per wave."""
    check(T, pos, spare, 8192, 2048, 40)


@pytest.mark.gpu
def test_conv_runs_of_8_tokens_few_channels():
    check(517, 3, 0, 1024, 256, 4)


def check(T, pos, spare, C, key_dim, Hv):
    g = torch.Generator(device=DEV)
    g.manual_seed(T + pos)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).bfloat16()
    proj, cw, R = r(T, C + 2 * Hv + 8), r(C, 4), T + 3 + spare
    ring = r(R, C)
    ring2 = ring.clone()
    got = conv(proj, ring, pos, cw, C, key_dim, Hv, C + 8)
    parts = [conv(proj[t:t + 8], ring2, pos + t, cw, C, key_dim, Hv, C + 8) for t in range(0, T, 8)]
    for a, b in zip(got, zip(*parts)):
        assert torch.equal(a.view(torch.int16), torch.cat(b).view(torch.int16))
    assert torch.equal(ring.view(torch.int16), ring2.view(torch.int16))
