"""Every block shape of the prefill GEMM at its edges (GPU): row counts around the
16-row fragments, the small kernel's limit (64) and the row blocks (64, 128),
output counts that end inside a tile, a wave or a column group (and, odd, take
the element stores), the shortest K and ring wrap-arounds, and rows and columns
that each shape is picked for. Against x @ W~^T in float64, W~ the
bf16-dequantized weight: |y - ref| <= 2^-8 |ref| (the output's rounding) +
2^-16 sum |x| |W~| (fp32 sums), as in tests/test_qgemm_gpu.py."""

import numpy as np
import pytest
import torch

from qvex import _C, kernels, synth
from qvex.kernels import _ptr, _stream
from test_qgemm_gpu import DEV
from test_qmv_gpu import _dequant_np, to_dev

SHAPES = [(16, 64, 256), (17, 301, 512), (32, 4097, 768), (33, 128, 2304), (48, 272, 1024), (49, 80, 256), (64, 65, 512),
          (65, 64, 256), (65, 16, 768), (100, 2049, 512), (127, 301, 256), (129, 1040, 1280), (130, 2048, 256),
          (300, 4096, 512), (512, 8192, 256), (511, 10240, 768), (512, 24576, 256), (513, 12352, 512), (1000, 640, 2560),
          # 128 x 256 blocks (two tiles per wave): a partial row block, the columns ending in a wave's first tile
          (129, 24592, 256), (200, 21861, 256),
          # 128 x 384 blocks (three tiles per wave): the same, ending in a wave's first and second tile
          (301, 24250, 256), (450, 24265, 256), (257, 24300, 512)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_packed_gemm_shapes(M, N, K):
    w, s, b = synth.qmv_weights(N, K, seed=21, tag=N + M)
    x = synth.qmv_x(M, K, seed=21, tag=M)
    packed = kernels.pack_w4(to_dev(w, torch.int32), to_dev(s, torch.bfloat16), to_dev(b, torch.bfloat16))
    out = torch.full((M * N + 1,), 7.0, dtype=torch.bfloat16, device=DEV)
    y = out[:M * N] if M % 2 else out[1:]                     # the second: only 2-byte aligned
    _C.call("qvex_w4g64_packed_gemm", _ptr(to_dev(x, torch.bfloat16)), _ptr(packed), _ptr(y), M, N, K, _stream())
    torch.cuda.synchronize()
    Wd = torch.from_numpy(synth.bf16_to_f32(_dequant_np(w, s, b)).astype(np.float64)).to(DEV)
    xf = torch.from_numpy(synth.bf16_to_f32(x).astype(np.float64)).to(DEV)
    ref = xf @ Wd.T
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -16 * (xf.abs() @ Wd.abs().T)
    err = (y.view(M, N).double() - ref).abs()
    print(f"M={M} N={N} K={K}: max err / bound {float((err / bound).max()):.3f}", flush=True)
    assert bool((err <= bound).all())
    assert float(out[M * N if M % 2 else 0]) == 7.0           # nothing past the result


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(4096, 512), (24576, 256), (301, 768)])
def test_packed_gemm_row_bits_over_shapes(N, K):
    """A row's bits are the same whichever shape its call takes."""
    w, s, b = synth.qmv_weights(N, K, seed=22)
    packed = kernels.pack_w4(to_dev(w, torch.int32), to_dev(s, torch.bfloat16), to_dev(b, torch.bfloat16))
    x = to_dev(synth.qmv_x(1024, K, seed=22), torch.bfloat16)
    full = kernels.packed_gemm(x, packed, N)
    for lo, hi in ((0, 16), (40, 90), (100, 164), (300, 812), (1000, 1024)):
        part = kernels.packed_gemm(x[lo:hi].contiguous(), packed, N)
        assert torch.equal(full[lo:hi].view(torch.int16), part.view(torch.int16)), (lo, hi)


@pytest.mark.gpu
@pytest.mark.parametrize("M,I", [(33, 264), (65, 512), (129, 1032), (512, 12288),
                                 # 128 x 128, 128 x 256 and 128 x 384 blocks, partial in rows and columns
                                 (100, 8200), (130, 12296), (200, 12288), (301, 12136), (450, 12288)])
def test_packed_gemm_swiglu_shapes(M, I):
    K = 512
    w, s, b = synth.qmv_weights(2 * I, K, seed=23, tag=M)
    x = to_dev(synth.qmv_x(M, K, seed=23, tag=M), torch.bfloat16)
    wt, st, bt = to_dev(w, torch.int32), to_dev(s, torch.bfloat16), to_dev(b, torch.bfloat16)
    fused = kernels.packed_gemm(x, kernels.pack_w4(wt, st, bt, swiglu=True), 2 * I, swiglu=True)
    gu = kernels.packed_gemm(x, kernels.pack_w4(wt, st, bt), 2 * I)
    h = torch.empty((M, I), dtype=torch.bfloat16, device=DEV)
    _C.call("qvex_swiglu", _ptr(gu), _ptr(h), M, I, _stream())
    torch.cuda.synchronize()
    assert torch.equal(fused.view(torch.int16), h.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(20, 100, 512), (64, 272, 1024), (70, 300, 512), (256, 6144, 256), (512, 24576, 256)])
def test_packed_gemm_large_scales(M, N, K):
    """Scales around 2^104 and of 2^116 (weights up to 2^120) beside ordinary ones: the
    result is finite, within the bound of the shapes above, and a row without such a
    scale has the bits it has alone. A scale that is infinite still gives what it is."""
    w, s, b = synth.qmv_weights(N, K, seed=24)
    s, b = synth.bf16_to_f32(s).copy(), synth.bf16_to_f32(b).copy()
    plain = kernels.pack_w4(to_dev(w, torch.int32), to_dev(synth.bf16_bits(s), torch.bfloat16),
                            to_dev(synth.bf16_bits(b), torch.bfloat16))
    big = np.arange(3, N, 7)
    for i, e in zip(range(4), (103, 104, 110, 116)):
        rows = big[i::4]
        s[rows, i % s.shape[1]] = np.float32(1.5 * 2.0 ** e)
        b[rows, i % s.shape[1]] = np.float32(-8.0 * 1.5 * 2.0 ** e)
    s16, b16 = synth.bf16_bits(s), synth.bf16_bits(b)
    x = synth.qmv_x(M, K, seed=24)
    xt = to_dev(x, torch.bfloat16)
    y = kernels.packed_gemm(xt, kernels.pack_w4(to_dev(w, torch.int32), to_dev(s16, torch.bfloat16),
                                                to_dev(b16, torch.bfloat16)), N)
    torch.cuda.synchronize()
    Wd = torch.from_numpy(synth.bf16_to_f32(_dequant_np(w, s16, b16)).astype(np.float64)).to(DEV)
    xf = torch.from_numpy(synth.bf16_to_f32(x).astype(np.float64)).to(DEV)
    ref = xf @ Wd.T
    bound = 2.0 ** -8 * ref.abs() + 2.0 ** -16 * (xf.abs() @ Wd.abs().T)
    assert bool(y.isfinite().all())
    assert bool(((y.double() - ref).abs() <= bound).all())
    same = np.setdiff1d(np.arange(N), big)
    assert torch.equal(y[:, same].view(torch.int16), kernels.packed_gemm(xt, plain, N)[:, same].view(torch.int16))
    s[big[0], 0] = np.inf
    y = kernels.packed_gemm(xt, kernels.pack_w4(to_dev(w, torch.int32), to_dev(synth.bf16_bits(s), torch.bfloat16),
                                                to_dev(b16, torch.bfloat16)), N)
    bad = ~y.isfinite()
    assert bool(bad[:, big[0]].all())
    bad[:, big[0]] = False
    assert not bool(bad.any())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [40, 200])
def test_packed_gemm_large_scales_swiglu(M):
    K, I = 512, 520
    w, s, b = synth.qmv_weights(2 * I, K, seed=25)
    s, b = synth.bf16_to_f32(s).copy(), synth.bf16_to_f32(b).copy()
    s[I + 5, 1], b[I + 5, 1] = 2.0 ** 110, -(2.0 ** 113)               # an up row
    wt, st, bt = to_dev(w, torch.int32), to_dev(synth.bf16_bits(s), torch.bfloat16), to_dev(synth.bf16_bits(b), torch.bfloat16)
    x = to_dev(synth.qmv_x(M, K, seed=25), torch.bfloat16)
    fused = kernels.packed_gemm(x, kernels.pack_w4(wt, st, bt, swiglu=True), 2 * I, swiglu=True)
    gu = kernels.packed_gemm(x, kernels.pack_w4(wt, st, bt), 2 * I)
    h = torch.empty((M, I), dtype=torch.bfloat16, device=DEV)
    _C.call("qvex_swiglu", _ptr(gu), _ptr(h), M, I, _stream())
    torch.cuda.synchronize()
    assert bool(fused.isfinite().all()) and torch.equal(fused.view(torch.int16), h.view(torch.int16))
