"""qvex_attention on prompt chunks (calls of 9 positions and more) against causal
softmax attention times sigmoid(gate) in float64, at the edges of its 64-row
blocks, 32-key blocks, units and groups of units, and with the extremes of the
scores; a row's bits depend neither on the call nor on a keys_per_split of 256 or more.

Bound: the output is rounded to bf16 (2^-8 |ref|), P is carried as two bf16 terms
(2^-16 relative) and the sums are fp32: |err| <= 2^-8 |ref| + 2^-14 sigmoid(gate) sum p |v| + 1e-6."""

import math

import pytest
import torch

from qvex import _C
from qvex.kernels import _ptr, _stream, kv_tile_k, kv_tile_v

DEV = "cuda:0"


def inputs(L, Hq, Hkv, D, pos0, seed, scale=1.0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    cap = (pos0 + L + 63) // 32 * 32
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    return ((scale * r(L, Hq, D)).bfloat16(), r(Hkv, cap, D).bfloat16(), r(Hkv, cap, D).bfloat16(),
            r(L, Hq * 2 * D).bfloat16())


def attention(q, k, v, gate, pos0, kps, spare=0):
    L, Hq, D = q.shape
    Hkv, cap = k.shape[:2]
    max_keys = cap if spare else pos0 + L
    pos = torch.tensor([pos0], dtype=torch.int32, device=DEV)
    out = torch.empty((L, Hq * D), dtype=torch.bfloat16, device=DEV)
    need = int(_C.lib().qvex_attn_workspace_bytes(L, Hq, Hkv, D, max_keys, kps))
    ws = torch.full(((need + 3) // 4,), float("nan"), dtype=torch.float32, device=DEV)
    kt, vt = kv_tile_k(k), kv_tile_v(v)
    _C.call("qvex_attention", _ptr(q), _ptr(kt), _ptr(vt), _ptr(pos), L, Hq, Hkv, D, cap, max_keys, max_keys, kps,
            _ptr(gate), gate.stride(0), _ptr(out), _ptr(ws), ws.numel() * 4, _stream())
    return out.view(L, Hq, D)


def reference(q, k, v, gate, pos0):
    L, Hq, D = q.shape
    Hkv = k.shape[0]
    rep = lambda t: t[:, :pos0 + L].double().repeat_interleave(Hq // Hkv, dim=0)
    s = torch.matmul(q.double().transpose(0, 1), rep(k).transpose(1, 2).contiguous()) / math.sqrt(D)
    seen = torch.arange(pos0 + L, device=DEV)[None] <= pos0 + torch.arange(L, device=DEV)[:, None]
    p = torch.softmax(s.masked_fill(~seen, -math.inf), dim=-1)
    sig = torch.sigmoid(gate.double().view(L, Hq, 2 * D)[..., D:])
    o = lambda x: torch.matmul(p, x).transpose(0, 1) * sig
    return o(rep(v)), o(rep(v).abs())


@pytest.mark.gpu
@pytest.mark.parametrize("L,Hq,Hkv,D,pos0,kps,spare", [
    (93, 16, 4, 256, 0, 512, 0), (96, 16, 4, 256, 31, 128, 0), (97, 16, 4, 256, 995, 512, 0),
    (190, 4, 2, 128, 33, 128, 1), (130, 6, 2, 128, 257, 256, 0), (117, 6, 2, 256, 1, 512, 0),
    (25, 16, 1, 128, 600, 128, 0), (370, 8, 8, 128, 5, 512, 1), (512, 16, 4, 256, 1536, 2048, 0),
    # 9 positions and up, one tile and part of a block
    (9, 16, 4, 256, 119, 128, 0), (9, 2, 2, 128, 0, 256, 0), (17, 16, 16, 256, 255, 256, 0), (65, 4, 1, 256, 511, 256, 1),
    # a group of four units per block: whole groups, a last one of one unit and of three, fewer than four units
    (512, 8, 8, 256, 1600, 128, 0), (512, 8, 8, 256, 1900, 128, 1), (300, 8, 8, 256, 3700, 128, 0),
    (520, 8, 8, 128, 3800, 128, 0), (2300, 16, 16, 256, 0, 1024, 0)])
def test_prefill_attention(L, Hq, Hkv, D, pos0, kps, spare):
    q, k, v, gate = inputs(L, Hq, Hkv, D, pos0, seed=L + pos0)
    got = attention(q, k, v, gate, pos0, kps, spare).double()
    ref, absref = reference(q, k, v, gate, pos0)
    ratio = ((got - ref).abs() / (2.0 ** -8 * ref.abs() + 2.0 ** -14 * absref + 1e-6)).max().item()
    print(f"worst ratio {ratio:.3f}")
    assert ratio <= 1.0


@pytest.mark.gpu
def test_prefill_attention_large_scores():
    """Scores of +-100 and growing along the keys: the reference moves many times."""
    q, k, v, gate = inputs(96, 16, 4, 256, 700, seed=3, scale=12.0)
    ramp = torch.linspace(0.2, 2.0, k.shape[1], device=DEV)[None, :, None]
    k = (k.float() * ramp).bfloat16()
    got = attention(q, k, v, gate, 700, 512).double()
    ref, absref = reference(q, k, v, gate, 700)
    # scores of magnitude S carry fp32 rounding of about 2^-21 S into the exponent
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -12 * absref + 1e-6).all()


@pytest.mark.gpu
def test_prefill_attention_rows_do_not_depend_on_the_call():
    q, k, v, gate = inputs(200, 16, 4, 256, 64, seed=4, scale=4.0)
    full = attention(q, k, v, gate, 64, 512)
    part = attention(q[:100].contiguous(), k, v, gate[:100].contiguous(), 64, 512)
    assert torch.equal(part.view(torch.int16), full[:100].view(torch.int16))


@pytest.mark.gpu
def test_prefill_attention_nan_key_reaches_only_the_rows_that_see_it():
    q, k, v, gate = inputs(96, 16, 4, 256, 100, seed=5)
    k[1, 150, 7] = float("nan")
    got = attention(q, k, v, gate, 100, 512).isnan()
    assert got[50:, 4:8].all()
    got[50:, 4:8] = False
    assert not got.any()


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,D,pos0,L,kps", [(16, 4, 256, 0, 90, 256), (16, 4, 256, 4000, 600, 256),
                                                 (8, 8, 256, 2011, 512, 128), (8, 8, 128, 4001, 500, 128)])
def test_prefill_attention_rows_over_block_forms(Hq, Hkv, D, pos0, L, kps):
    """Parts that start inside a tile, a block of keys and a unit; the whole takes a
    group of units per block (the last three), the parts one unit."""
    q, k, v, gate = inputs(L, Hq, Hkv, D, pos0, seed=6, scale=4.0)
    full = attention(q, k, v, gate, pos0, kps)
    for lo, n in ((0, 9), (1, 16), (7, 33), (L - 70, 70)):
        part = attention(q[lo:lo + n].contiguous(), k, v, gate[lo:lo + n].contiguous(), pos0 + lo, kps, spare=lo % 2)
        assert torch.equal(part.view(torch.int16), full[lo:lo + n].view(torch.int16)), (lo, n)
    if kps == 256:
        assert torch.equal(attention(q, k, v, gate, pos0, 2048).view(torch.int16), full.view(torch.int16))


def test_attention_workspace_serves_smaller_calls():
    """The size never falls as a call grows, and a record per unit is its upper bound."""
    size = _C.lib().qvex_attn_workspace_bytes
    for Hq, Hkv, D in ((16, 4, 256), (8, 8, 128), (16, 1, 256), (8, 2, 128)):
        QT = 16 // (Hq // Hkv)
        for kps in (128, 256, 2048):
            prev = {}
            for L in (1, 8, 9, 17, 64, 100, 512, 1000):
                last = 0
                for keys in (1, 128, 129, 1000, 4096, 5000, 20000, 131072):
                    n = int(size(L, Hq, Hkv, D, keys, kps))
                    assert n >= last and n >= prev.get(keys, 0), (Hq, Hkv, D, kps, L, keys)
                    assert n <= Hkv * -(-L // QT) * -(-keys // (kps if L < 9 else min(kps, 256))) * 16 * (D + 2) * 4
                    prev[keys] = last = n


@pytest.mark.gpu
@pytest.mark.parametrize("pos0,L", [(100, 40), (2011, 512)])
def test_prefill_attention_nan_query_stays_in_its_row(pos0, L):
    """A row of NaN scores is NaN as softmax attention has it, whatever unit it falls in;
    its tile's other rows keep their bits."""
    q, k, v, gate = inputs(L, 8, 8, 256, pos0, seed=7)
    clean = attention(q, k, v, gate, pos0, 128)
    q[19, 3, 5] = float("nan")
    got = attention(q, k, v, gate, pos0, 128)
    assert got[19, 3].isnan().all()
    got[19, 3] = clean[19, 3]
    assert torch.equal(got.view(torch.int16), clean.view(torch.int16))
