"""The matrix-vector kernel (weights [out, in], one to four token rows): feature counts on both sides of what its blocks of one to twelve
waves take in a round, rows of one group of k-steps and of several, padded weight rows, the non-temporal and the plain loads, and token
rows that take most of the LDS.  Tolerance, element by element: the products of halves are exact in fp32, a sum of K of them is off by at
most K 2^-23 of the sum of magnitudes in any order, and the result is rounded once to fp16."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(M, N, K, pad=0):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K + M)
    X = torch.randn(M, K, device="cuda", generator=gen, dtype=torch.float16)
    W = torch.randn(N, K + pad, device="cuda", generator=gen, dtype=torch.float16)[:, :K]
    return X, W


def _close(Y, X, W):
    ref, mag = X.double() @ W.double().T, X.double().abs() @ W.double().abs().T
    return bool(((Y.double() - ref).abs() <= 2.0 ** -11 * ref.abs() + X.shape[1] * 2.0 ** -23 * mag + 2.0 ** -25).all())


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K,pad", [(256, 2048, 0), (260, 4096, 8), (2044, 2048, 0), (2052, 6144, 0), (3076, 2048, 16), (5120, 2048, 0), (2820, 14336, 0), (260, 20480, 0)])
def test_any_number_of_features(dev, M, N, K, pad):
    X, W = _inputs(M, N, K, pad)
    Y = torch.full((M + 1, N), 7.0, device="cuda", dtype=torch.float16)
    dev.call("lg_gemm_f16", 1, 0, N, M, K, W.data_ptr(), K + pad, X, K, Y, N)
    dev.sync()
    assert _close(Y[:M], X, W)
    assert bool((Y[M] == 7.0).all())
    alone = torch.empty(M, (N + 7) // 8 * 8, device="cuda", dtype=torch.float16)
    for m in range(M):      # a row's bits do not depend on the other rows (outputs 16-byte aligned, as the kernel wants them)
        dev.call("lg_gemm_f16", 1, 0, N, 1, K, W.data_ptr(), K + pad, X.data_ptr() + 2 * m * K, K, alone[m].data_ptr(), N)
    dev.sync()
    assert torch.equal(Y[:M], alone[:, :N])


@pytest.mark.parametrize("M,N,K", [(1, 264, 2048), (3, 1032, 4096), (4, 4104, 2048)])
def test_members_of_a_group_have_the_bits_of_single_calls(dev, M, N, K):
    X, W = _inputs(M, 3 * N, K)
    Y, Z = (torch.empty(3, M, N, device="cuda", dtype=torch.float16) for _ in range(2))
    pointers = lambda t, step: (C.c_void_p * 3)(*[t.data_ptr() + 2 * i * step for i in range(3)])
    ldc = (C.c_int * 3)(N, N, N)
    dev.call("lg_gemm_fused_grouped_f16", 1, N, M, K, 3, pointers(W, N * K), K, X, K, pointers(Y, M * N), ldc, 0, None, 0, 0, 0)
    for i in range(3):
        dev.call("lg_gemm_f16", 1, 0, N, M, K, W.data_ptr() + 2 * i * N * K, K, X, K, Z.data_ptr() + 2 * i * M * N, N)
    dev.sync()
    assert torch.equal(Y, Z)
    assert _close(Y.transpose(0, 1).reshape(M, 3 * N), X, W)
