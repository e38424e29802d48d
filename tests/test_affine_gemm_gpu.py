"""qvex_affine_gemm: the any-width product on prompt chunks, against the float64
oracle with the bound of the 1..8-row kernel (|err| <= 2^-8 |ref| + 2^-14 sum|x| (|s| q + |b|):
the same fp32 sums of exact codes, one bf16 rounding), at the edges of its row
blocks, output tiles and 128-code stages; a row's bits do not depend on M."""

import ctypes

import pytest
import torch

from qvex import _C, kernels, synth
from qvex.model import QLinear
from test_affine_gpu import bits16, check, to_dev, weights


def product(x, w, s, b, bits, gs):
    return kernels.quantized_matmul_affine(to_dev(x, torch.bfloat16), to_dev(w, torch.int32),
                                           to_dev(s, torch.bfloat16), to_dev(b, torch.bfloat16), gs, bits, gemm=True)


@pytest.mark.gpu
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bits", [2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("M,N,stages", [(1, 1, 1), (16, 65, 3), (33, 63, 2), (65, 130, 2)])
def test_affine_gemm_vs_oracle(M, N, stages, bits, gs):
    K = 128 * stages - (128 - gs if gs < 128 else 0)      # a last stage of one group
    w, s, b, _ = weights(N, K, bits, gs, seed=bits * 100 + gs + M)
    x = synth.qmv_x(M, K, seed=21, tag=bits)
    y = product(x, w, s, b, bits, gs)
    torch.cuda.synchronize()
    check(x, w, s, b, bits, gs, bits16(y))


@pytest.mark.gpu
@pytest.mark.parametrize("bits,gs", [(8, 64), (5, 32), (4, 64)])
def test_affine_gemm_rows_do_not_depend_on_the_call(bits, gs):
    """16-, 32- and 64-row blocks (M = 16, 50, 600 at 4096 outputs)."""
    N, K = 4096, 448
    w, s, b, _ = weights(N, K, bits, gs, seed=bits)
    x = synth.qmv_x(600, K, seed=22)
    full = product(x, w, s, b, bits, gs)
    for m in (16, 50):
        part = product(x[:m], w, s, b, bits, gs)
        assert torch.equal(part.view(torch.int16), full[:m].view(torch.int16))
    torch.cuda.synchronize()
    check(x[:64], w, s, b, bits, gs, bits16(full[:64]))


@pytest.mark.parametrize("M,N,K,bits,gs", [(0, 16, 128, 8, 64), (16, 0, 128, 8, 64), (16, 16, 96, 8, 64),
                                           (16, 16, 0, 8, 64), (16, 16, 128, 7, 64), (16, 16, 128, 8, 16)])
def test_affine_gemm_rejects(M, N, K, bits, gs):
    p16 = (ctypes.addressof(ctypes.create_string_buffer(64)) + 15) // 16 * 16
    with pytest.raises(_C.QvexError, match="qvex_affine_gemm"):
        _C.call("qvex_affine_gemm", p16, p16, p16, p16, p16, M, N, K, bits, gs, None)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,bits,gs,chunks", [
    (16, 130, 8256, 4, 64, True), (48, 512, 12352, 4, 64, True), (40, 1024, 12352, 4, 64, False),
    (63, 65, 12352, 4, 64, True), (64, 65, 12352, 4, 64, False), (16, 4096, 4160, 4, 64, False), (16, 130, 1088, 4, 64, False),
    (16, 512, 8192, 5, 64, True), (17, 512, 8192, 5, 64, True), (24, 512, 8192, 5, 64, False), (16, 64, 8256, 8, 64, False), (16, 64, 12288, 8, 64, True),
    (16, 2050, 8192, 6, 32, False), (24, 64, 12288, 3, 32, True), (32, 64, 12288, 3, 32, False), (15, 96, 448, 8, 64, True)])
def test_unpacked_layer_takes_chunks_or_gemm(M, N, K, bits, gs, chunks):
    """Either side of the rule that leaves a short call of a long, narrow layer to
    chunks of 8 rows: the bits are those of the path it names, within the oracle's bound."""
    w, s, b, _ = weights(N, K, bits, gs, seed=N + K)
    x = synth.qmv_x(M, K, seed=23)
    wt, st, bt = to_dev(w, torch.int32), to_dev(s, torch.bfloat16), to_dev(b, torch.bfloat16)
    xt = to_dev(x, torch.bfloat16)
    y = QLinear(wt, st, bt, gs, bits)(xt)
    if chunks:
        ref = torch.cat([kernels.quantized_matmul(xt[m:m + 8], wt, st, bt, group_size=gs, bits=bits)
                         for m in range(0, M, 8)])
    else:
        ref = kernels.quantized_matmul_affine(xt, wt, st, bt, gs, bits, gemm=True)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
    check(x, w, s, b, bits, gs, bits16(y))
