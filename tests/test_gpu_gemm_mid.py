"""The tiles fitted to the token count (gemm_mid.hpp): heights and widths at their edges, K-slices that meet inside the kernel, every
layout and epilogue, streams with and without a workspace.  Tolerances are those of the other GEMM tests: one fp16 rounding of an
fp32 sum (2^-11 of the value, 5e-4 of the largest) and the summation order."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.conftest import max_rel_err

pytestmark = pytest.mark.gpu

TILED = 2


def rnd(po, n, tid, std=1.0):
    return po.fill_normal(n, 0, tid, 0.0, std, 1)


def weight(dev, W, layout):
    """W [K, N] (numpy) as the device matrix of a layout and its leading dimension"""
    K, N = W.shape
    if layout == 0:
        return dev.up(W, 1), N
    plain = dev.up(np.ascontiguousarray(W.T), 1)
    if layout == 1:
        return plain, K
    t = dev.empty((N * K,), 1)
    dev.call("lg_weight_tile_f16", t, plain, N, K, 1, K)
    dev.sync()
    return t, K


# token counts on both sides of every tile height; features that only one of the widths 96 / 128 / 192 / 256 divides and that
# several do; K of one k-tile, of fewer k-tiles than a ring holds, and long enough for two and for eight slices
@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [(1, 128, 64), (5, 128, 4096), (17, 384, 2048), (32, 256, 192), (33, 640, 320), (64, 896, 1024), (65, 128, 4096), (96, 288, 256),
                                   (97, 768, 2048), (129, 1024, 1024), (160, 192, 1088), (161, 576, 2048), (193, 4096, 1024), (225, 2304, 448), (256, 512, 8192),
                                   (257, 1536, 2048), (320, 12288, 128), (511, 2048, 1024), (513, 3072, 256), (700, 6144, 128)])
def test_gemm_at_the_edges_of_the_tiles(dev, po, layout, M, N, K):
    X, W = rnd(po, M * K, 11).reshape(M, K), rnd(po, K * N, 12, 0.05).reshape(K, N)
    dW, ld = weight(dev, W, layout)
    dX, dY = dev.up(X, 1), dev.empty((M + 1, N), 1)
    dY.fill_(7.0)
    dev.call("lg_gemm_f16", layout, 0, N, M, K, dW, ld, dX, K, dY, N)
    got = dev.down(dY)
    assert np.all(got[M] == 7.0)
    assert max_rel_err(got[:M], po.gemm(X, W, 1)) < 2e-3
    # the counters at which K-slices meet are back where they were, and the slices are summed in one order: the same bits again
    for _ in range(3):
        dY.fill_(0.0)
        dev.call("lg_gemm_f16", layout, 0, N, M, K, dW, ld, dX, K, dY, N)
        assert np.array_equal(dev.down(dY)[:M], got[:M])


# fewer k-tiles than a ring is deep, as many and more, even and odd: loads go out for pairs of k-tiles, and the loop may end in either half of one
@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,N", [(20, 768), (96, 3072), (190, 6144), (250, 12288), (384, 3072), (500, 4608), (1100, 3072)])
def test_every_number_of_k_tiles(dev, po, layout, M, N):
    K = 13 * 64
    X, W = rnd(po, M * K, 13).reshape(M, K), rnd(po, K * N, 14, 0.05).reshape(K, N)
    dX = dev.up(X, 1)
    for kt in (1, 2, 3, 4, 5, 6, 7, 8, 13):
        k = 64 * kt
        dW, ld = weight(dev, np.ascontiguousarray(W[:k]), layout)
        dY = dev.empty((M, N), 1)
        dev.call("lg_gemm_f16", layout, 0, N, M, k, dW, ld, dX, K, dY, N)
        ref = (torch.from_numpy(X[:, :k]).cuda().float() @ torch.from_numpy(W[:k]).cuda().float()).cpu().numpy()
        assert max_rel_err(dev.down(dY), ref) < 2e-3, kt


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,S,h,d", [(72, 24, 8, 128), (90, 45, 8, 96), (130, 65, 16, 12), (48, 1, 32, 128), (300, 300, 6, 64)])
def test_fused_epilogues(dev, po, layout, M, S, h, d):
    """Bias, bias + GELU, GeGLU and the head-transposed store (whole rows of 16 bytes, and a head size that allows only 8) with K
    long enough to be sliced."""
    N, K, B = h * d, 2048, M // S
    if N % 192 and N % 128:
        pytest.skip("no tile divides the features")
    X, W, bias = rnd(po, M * K, 21).reshape(M, K), rnd(po, K * N, 22, 0.05).reshape(K, N), rnd(po, N, 23, 0.3)
    dW, ld = weight(dev, W, layout)
    dX, dB = dev.up(X, 1), dev.up(bias, 1)
    y = po.gemm(X, W, 1)
    for epi, ref in ((dev.capi.EPI_BIAS, po.round_f16(y + bias)), (dev.capi.EPI_BIAS_GELU, po.add_bias_gelu(y.copy(), bias, 1))):
        out = dev.empty((M, N + 4), 1)   # rows that are not 16-byte aligned
        out.fill_(7.0)
        dev.call("lg_gemm_fused_f16", layout, N, M, K, dW, ld, dX, K, out, N + 4, epi, dB, 0, 0, 0)
        got = dev.down(out)
        assert max_rel_err(got[:, :N], ref) < 4e-3 and np.all(got[:, N:] == 7.0)
    rows = S + 3
    ref, _, _ = po.add_qkv_bias_transpose(y, bias, y, bias, y, bias, B, S, h, d, 1)
    out = dev.empty((B, h, rows, d), 1)
    out.fill_(7.0)
    dev.call("lg_gemm_fused_f16", layout, N, M, K, dW, ld, dX, K, out, rows, dev.capi.EPI_BIAS_HEADS, dB, S, d, h)
    got = dev.down(out)
    assert max_rel_err(got[:, :, :S], ref) < 2e-3 and np.all(got[:, :, S:] == 7.0)
    idx = np.arange(N)
    idx = (idx // 32) * 16 + idx % 16 + np.where(idx % 32 >= 16, N // 2, 0)
    dG, ld = weight(dev, np.ascontiguousarray(W[:, idx]), layout)
    out = dev.empty((M, N // 2), 1)
    dev.call("lg_gemm_fused_f16", layout, N, M, K, dG, ld, dX, K, out, N // 2, 5, dev.up(bias[idx], 1), 0, 0, 0)
    assert max_rel_err(dev.down(out), po.add_bias_geglu(y, bias, 1)) < 4e-3


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,K", [(9, 2048), (64, 1024), (120, 4096), (400, 2048)])
def test_group_equals_plain_calls_bit_for_bit(dev, po, layout, M, K):
    """Q, K and V as one call and as three: how K is sliced must not depend on it.  (At 5-64 rows with weights [out, in] the
    weight-streaming kernel may take the group: equal up to the summation order.)"""
    h, d = 32, 128
    N = h * d
    S = 1 if M <= 64 else M
    B = M // S
    X = rnd(po, M * K, 31).reshape(M, K)
    dX = dev.up(X, 1)
    Ws, bs = [rnd(po, K * N, 32 + t, 0.05).reshape(K, N) for t in range(3)], [rnd(po, N, 35 + t, 0.3) for t in range(3)]
    pairs = [weight(dev, W, layout) for W in Ws]
    dB = [dev.up(b, 1) for b in bs]
    arr = lambda ptrs: (C.c_void_p * 3)(*ptrs)
    plain, grouped = [dev.empty((B, h, S, d), 1) for _ in range(3)], [dev.empty((B, h, S, d), 1) for _ in range(3)]
    for t in range(3):
        dev.call("lg_gemm_fused_f16", layout, N, M, K, pairs[t][0], pairs[t][1], dX, K, plain[t], S, dev.capi.EPI_BIAS_HEADS, dB[t], S, d, h)
    dev.call("lg_gemm_fused_grouped_f16", layout, N, M, K, 3, arr([p[0].data_ptr() for p in pairs]), pairs[0][1], dX, K, arr([g.data_ptr() for g in grouped]),
             (C.c_int * 3)(S, S, S), dev.capi.EPI_BIAS_HEADS, arr([b.data_ptr() for b in dB]), S, d, h)
    for t in range(3):
        got, ref = dev.down(grouped[t]), dev.down(plain[t])
        if M > 64 or layout == 0:
            assert np.array_equal(got, ref)
        else:
            assert max_rel_err(got, ref) < 1e-3
        want, _, _ = po.add_qkv_bias_transpose(po.gemm(X, Ws[t], 1), bs[t], po.gemm(X, Ws[t], 1), bs[t], po.gemm(X, Ws[t], 1), bs[t], B, S, h, d, 1)
        assert max_rel_err(got, want) < 2e-3


def test_streams_of_their_own_and_a_stream_without_a_workspace(dev, po):
    """Sliced GEMMs in flight on two streams at the same time use two workspaces; a stream the library does not know has none and
    K is not sliced on it."""
    M, N, K = 200, 2048, 4096
    X = [rnd(po, M * K, 41 + i).reshape(M, K) for i in range(2)]
    W = rnd(po, K * N, 43, 0.05).reshape(K, N)
    dW, ld = weight(dev, W, TILED)
    dX = [dev.up(x, 1) for x in X]
    ref = []
    for x in dX:
        y = dev.empty((M, N), 1)
        dev.call("lg_gemm_f16", TILED, 0, N, M, K, dW, ld, x, K, y, N)
        ref.append(dev.down(y))
    streams = []
    for _ in range(2):
        p = C.c_void_p()
        assert dev.lib.lg_stream_create(C.byref(p)) == 0
        streams.append(p)
    outs = [[dev.empty((M, N), 1) for _ in range(20)] for _ in range(2)]
    dev.sync()
    for r in range(20):
        for i in range(2):
            assert dev.lib.lg_gemm_f16(TILED, 0, N, M, K, dW.data_ptr(), ld, dX[i].data_ptr(), K, outs[i][r].data_ptr(), N, streams[i]) == 0
    dev.sync()
    for i in range(2):
        for y in outs[i]:
            assert np.array_equal(dev.down(y), ref[i])
        assert dev.lib.lg_stream_destroy(streams[i]) == 0
    other = torch.cuda.Stream()
    y = dev.empty((M, N), 1)
    dev.sync()
    assert dev.lib.lg_gemm_f16(TILED, 0, N, M, K, dW.data_ptr(), ld, dX[0].data_ptr(), K, y.data_ptr(), N, C.c_void_p(other.cuda_stream)) == 0
    dev.sync()
    assert max_rel_err(dev.down(y), ref[0]) < 1e-3


@pytest.mark.parametrize("layout", [1, 2])
@pytest.mark.parametrize("M,N,K", [(70, 3072, 960), (106, 1920, 2048), (200, 6144, 1088), (240, 12288, 1024), (256, 11264, 1024), (384, 4608, 1024), (511, 2304, 4096)])
def test_turned_loops(dev, po, layout, M, N, K):
    """Feature blocks of 768 that start at different k-tiles (from 16 k-tiles on): fewer k-tiles than the turns add up to, a last block that is not whole,
    K-slices; and a member of a group of three has the bits of a call of its own, whichever tiles the two take."""
    X = rnd(po, M * K, 21).reshape(M, K)
    Ws = [rnd(po, K * N, 22 + i, 0.05).reshape(K, N) for i in range(3)]
    dX, bias = dev.up(X, 1), dev.up(rnd(po, N, 25), 1)
    dW = [weight(dev, W, layout)[0] for W in Ws]
    one = [dev.empty((1, N // 128, M, 128), 1) for _ in range(3)]
    for i in range(3):
        dev.call("lg_gemm_fused_f16", layout, N, M, K, dW[i], K, dX, K, one[i], M, dev.capi.EPI_BIAS_HEADS, bias, M, 128, 0)
    three = [dev.empty((1, N // 128, M, 128), 1) for _ in range(3)]
    ptrs = lambda ts: (C.c_void_p * 3)(*[t.data_ptr() for t in ts])
    dev.call("lg_gemm_fused_grouped_f16", layout, N, M, K, 3, ptrs(dW), K, dX, K, ptrs(three), (C.c_int * 3)(M, M, M), dev.capi.EPI_BIAS_HEADS, ptrs([bias] * 3), M, 128, 0)
    want = [po.gemm(X, W, 1) + dev.down(bias) for W in Ws]
    for i in range(3):
        got = dev.down(one[i])
        assert np.array_equal(got, dev.down(three[i]))
        assert max_rel_err(got[0].transpose(1, 0, 2).reshape(M, N), want[i]) < 2e-3


# on both sides of 512 rows and of 3 145 728 outputs, K long enough for slices; one block of 768 features and several
@pytest.mark.parametrize("M,N,K", [(257, 1536, 2048), (300, 3072, 2048), (511, 2304, 4096), (513, 2304, 2048), (700, 4096, 2048), (768, 4096, 2048), (1024, 1024, 4096)])
def test_above_256_rows_a_row_does_not_depend_on_its_call(dev, po, M, N, K):
    """One sum in the order of k whatever computes it: a range of the rows (more than 256 of them), a range of the features and the
    three layouts have the bits of the whole call."""
    X, W = rnd(po, M * K, 51).reshape(M, K), rnd(po, K * N, 52, 0.05).reshape(K, N)
    dX = dev.up(X, 1)
    first = None
    for layout in (0, 1, 2):
        dW, ld = weight(dev, W, layout)

        def gemm(rows, r0, n, n0):
            y = dev.empty((rows, n), 1)
            dev.call("lg_gemm_f16", layout, 0, n, rows, K, dW.data_ptr() + 2 * n0 * (1 if layout == 0 else K), ld, dX.data_ptr() + 2 * r0 * K, K, y, n)
            return dev.down(y)

        whole = gemm(M, 0, N, 0)
        first = whole if layout == 0 else first
        assert np.array_equal(whole, first)
        assert np.array_equal(gemm(257, M - 257, N, 0), whole[M - 257:])
        for n0 in (256, 768):
            assert np.array_equal(gemm(M, 0, N - n0, n0), whole[:, n0:]) and np.array_equal(gemm(M, 0, n0, 0), whole[:, :n0])
    assert max_rel_err(first, po.gemm(X, W, 1)) < 2e-3


def test_on_a_stream_with_half_of_the_compute_units(dev, po):
    """The plans are made for the units of the stream: above 256 rows the bits are those of the whole chip, up to 256 K is sliced
    another way, always the same one."""
    N, K = 3072, 4096
    W = rnd(po, K * N, 53, 0.05).reshape(K, N)
    dW, ld = weight(dev, W, TILED)
    s = C.c_void_p()
    assert dev.lib.lg_stream_create_cu_mask(C.byref(s), (C.c_uint * 8)(*[0xFFFFFFFF] * 4 + [0] * 4), 8) == 0, dev.capi.last_error()
    try:
        for M in (40, 200, 300):
            X = rnd(po, M * K, 54 + M).reshape(M, K)
            dX, whole = dev.up(X, 1), dev.empty((M, N), 1)
            dev.call("lg_gemm_f16", TILED, 0, N, M, K, dW, ld, dX, K, whole, N)
            outs = [dev.empty((M, N), 1) for _ in range(4)]
            dev.sync()
            for y in outs:
                assert dev.lib.lg_gemm_f16(TILED, 0, N, M, K, dW.data_ptr(), ld, dX.data_ptr(), K, y.data_ptr(), N, s) == 0
            got = [dev.down(y) for y in outs]
            assert all(np.array_equal(g, got[0]) for g in got)
            assert max_rel_err(got[0], po.gemm(X, W, 1)) < 2e-3
            if M > 256:
                assert np.array_equal(got[0], dev.down(whole))
    finally:
        assert dev.lib.lg_stream_destroy(s) == 0


# 256-row tiles in rounds of 16, 8 and 4 rows of tiles, a last round that is not whole and no rounds; lower tiles in more than one round
@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,N", [(4000, 2048), (2048, 4096), (1024, 8192), (5000, 6144), (5000, 3072), (2500, 8192), (1536, 12288)])
def test_placement_on_the_xcds(dev, layout, M, N):
    """Every tile is computed, whichever workgroups do it: on the whole chip and on a stream with half of it, whose rounds are half as large."""
    K = 192
    gen = torch.Generator(device="cuda")
    gen.manual_seed(8)
    X, W = torch.randn(M, K, device="cuda", generator=gen).half(), (0.05 * torch.randn(K, N, device="cuda", generator=gen)).half()
    ref, w, ld = X.float() @ W.float(), W, N
    if layout:
        w, ld = W.t().contiguous(), K
    if layout == TILED:
        plain, w = w, torch.empty_like(w)
        dev.call("lg_weight_tile_f16", w, plain, N, K, 1, K)
    s, ys = C.c_void_p(), [torch.full((M, N), 7e4, device="cuda", dtype=torch.float32).half() for _ in range(2)]
    assert dev.lib.lg_stream_create_cu_mask(C.byref(s), (C.c_uint * 8)(*[0xFFFFFFFF] * 4 + [0] * 4), 8) == 0, dev.capi.last_error()
    try:
        dev.sync()
        for y, stream in zip(ys, (C.c_void_p(dev.stream), s)):
            assert dev.lib.lg_gemm_f16(layout, 0, N, M, K, w.data_ptr(), ld, X.data_ptr(), K, y.data_ptr(), N, stream) == 0
            dev.sync()
            assert float((y.float() - ref).abs().max()) < 2e-3 * float(ref.abs().max())
    finally:
        assert dev.lib.lg_stream_destroy(s) == 0
    assert torch.equal(*ys)


# 128 x 192 tiles with weights [in, out] above 256 rows have an order of the loads of their own: fewer k-tiles than a ring is deep, as many and more
@pytest.mark.parametrize("M,N", [(389, 12288), (512, 12288), (978, 6144)])
def test_128_x_192_tiles_of_in_out_weights(dev, M, N):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    for K in (64, 128, 192, 256, 320, 384, 576, 1088):
        X, W = torch.randn(M, K, device="cuda", generator=gen).half(), (0.05 * torch.randn(K, N, device="cuda", generator=gen)).half()
        t, Y = W.t().contiguous(), [torch.full((M, N), 7e4, device="cuda", dtype=torch.float32).half() for _ in range(2)]
        torch.cuda.synchronize()
        dev.call("lg_gemm_f16", 0, 0, N, M, K, W.data_ptr(), N, X.data_ptr(), K, Y[0].data_ptr(), N)
        dev.call("lg_gemm_f16", 1, 0, N, M, K, t.data_ptr(), K, X.data_ptr(), K, Y[1].data_ptr(), N)
        dev.sync()
        ref = X.float() @ W.float()
        assert float((Y[0].float() - ref).abs().max()) < 2e-3 * float(ref.abs().max())
        assert torch.equal(*Y)
