"""Which launches a GEMM call makes, read from a graph that the call is captured into: calls that one kernel can take must not fall
through to slower ways (a second kernel, a kernel on a fraction of the chip, a call for every token row)."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.conftest import max_rel_err

pytestmark = pytest.mark.gpu


class _KernelNode(C.Structure):
    _fields_ = [("block", C.c_uint * 3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", C.c_uint * 3), ("params", C.c_void_p), ("shared", C.c_uint)]


@pytest.fixture
def stream(dev):
    p = C.c_void_p()
    assert dev.lib.lg_stream_create(C.byref(p)) == 0
    yield p
    assert dev.lib.lg_stream_destroy(p) == 0


def launches(dev, stream, name, *args, replays=1, between=None):
    """[workgroups] of the kernels that the call launches; the graph is then run, with `between` after each replay."""
    hip, graph, run = dev.lib, C.c_void_p(), C.c_void_p()   # the HIP runtime that the library itself uses
    dev.sync()
    assert hip.hipStreamBeginCapture(stream, 0) == 0
    rc = getattr(dev.lib, name)(*[C.c_void_p(a.data_ptr()) if hasattr(a, "data_ptr") else a for a in args], stream)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0, dev.capi.last_error()
    n = C.c_size_t()
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    nodes, out = (C.c_void_p * n.value)(), []
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(n)) == 0
    for node in nodes:
        p = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)) == 0
        out.append(p.grid[0] * p.grid[1] * p.grid[2])
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
    for _ in range(replays):
        assert hip.hipGraphLaunch(run, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
        if between:
            between()
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    return out


def rnd(po, n, tid, std=1.0):
    return po.fill_normal(n, 0, tid, 0.0, std, 1)


def weight(dev, W, layout):
    """W [N, K] as the device matrix of layout 0 ([in, out]), 1 ([out, in]) or 2 (fragment blocks)"""
    plain = dev.up(np.ascontiguousarray(W.T) if layout == 0 else W, 1)
    if layout != 2:
        return plain
    t = dev.empty((W.size,), 1)
    dev.call("lg_weight_tile_f16", t, plain, W.shape[0], W.shape[1], 1, W.shape[1])
    dev.sync()
    return t


# features that are a multiple of neither 96 nor 128, on both sides of the row count from which the tile kernels are preferred
@pytest.mark.parametrize("layout", [1, 2])
@pytest.mark.parametrize("M", [48, 49, 64])
def test_features_no_tile_divides_stay_on_one_launch(dev, po, stream, layout, M):
    N, K = 8224, 2048
    X, W = rnd(po, M * K, 61).reshape(M, K), rnd(po, N * K, 62, 0.05).reshape(N, K)
    dX, dW, y = dev.up(X, 1), weight(dev, W, layout), dev.empty((M, N), 1)
    got = launches(dev, stream, "lg_gemm_f16", layout, 0, N, M, K, dW, K, dX, K, y, N)
    assert len(got) == 1 and got[0] >= 128
    assert max_rel_err(dev.down(y), po.gemm(X, np.ascontiguousarray(W.T), 1)) < 2e-3


@pytest.mark.parametrize("layout", [1, 2])
@pytest.mark.parametrize("M", [48, 49, 64])
def test_projections_with_row_places_stay_on_one_launch(dev, po, stream, layout, M):
    N, K, d = 2912, 2048, 32
    h = N // d
    X = rnd(po, M * K, 63).reshape(M, K)
    Ws, bs = [rnd(po, N * K, 64 + i, 0.05).reshape(N, K) for i in range(3)], [rnd(po, N, 67 + i, 0.3) for i in range(3)]
    dX, dW, dB = dev.up(X, 1), [weight(dev, W, layout) for W in Ws], [dev.up(b, 1) for b in bs]
    out = [dev.empty((M, h, 1, d), 1) for _ in range(3)]
    ptrs, ints = lambda ts: (C.c_void_p * 3)(*[t.data_ptr() for t in ts]), lambda v: (C.c_int * len(v))(*v)
    slots = [(5 * r + 3) % M if M % 5 else M - 1 - r for r in range(M)]
    got = launches(dev, stream, "lg_gemm_fused_grouped_rows_f16", layout, N, M, K, 3, ptrs(dW), K, dX, K, ptrs(out), ints([1, 1, 1]), ptrs(dB), d, h,
                   ints([0, 1, 1]), ints(slots), ints([0] * M))
    assert len(got) == 1 and got[0] >= 128
    for i in range(3):
        ref = po.round_f16(po.gemm(X, np.ascontiguousarray(Ws[i].T), 1) + bs[i]).reshape(M, h, 1, d)
        res = dev.down(out[i])
        assert max_rel_err(res[slots] if i else res, ref) < 2e-3


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [(11, 4096, 4096), (48, 3072, 4096), (64, 4096, 4096), (106, 4096, 2048), (200, 2048, 2048)])
def test_a_member_alone_has_the_chip_and_the_bits_of_its_group(dev, po, stream, layout, M, N, K):
    """How K is sliced does not depend on how many members come together: as one of three a member has the bits it has alone (except
    where the weight-streaming kernel takes the three), and alone it has as many workgroups as a plain call, a projection (whose slices
    have to suit three as well) a third of them at least."""
    d = 128
    X = rnd(po, M * K, 71).reshape(M, K)
    Ws, bs = [rnd(po, N * K, 72 + i, 0.05).reshape(N, K) for i in range(3)], [rnd(po, N, 75 + i, 0.3) for i in range(3)]
    dX, dW, dB = dev.up(X, 1), [weight(dev, W, layout) for W in Ws], [dev.up(b, 1) for b in bs]
    ld = N if layout == 0 else K
    ptrs = lambda ts: (C.c_void_p * 3)(*[t.data_ptr() for t in ts])
    plain = launches(dev, stream, "lg_gemm_f16", layout, 0, N, M, K, dW[0], ld, dX, K, dev.empty((M, N), 1), N)
    for epi, a0, a1, ldc in ((dev.capi.EPI_BIAS_HEADS, 1, d, 1), (dev.capi.EPI_BIAS, 0, 0, N), (dev.capi.EPI_BIAS_GELU, 0, 0, N)):
        one, three = [[dev.empty((M, N), 1) for _ in range(3)] for _ in range(2)]
        for i in range(3):
            got = launches(dev, stream, "lg_gemm_fused_f16", layout, N, M, K, dW[i], ld, dX, K, one[i], ldc, epi, dB[i], a0, a1, 0)
            assert len(got) == len(plain) and 3 * got[0] >= plain[0] and (epi == dev.capi.EPI_BIAS_HEADS or got == plain)
        launches(dev, stream, "lg_gemm_fused_grouped_f16", layout, N, M, K, 3, ptrs(dW), ld, dX, K, ptrs(three), (C.c_int * 3)(ldc, ldc, ldc), epi, ptrs(dB), a0, a1, 0)
        for i in range(3):
            got, ref = dev.down(three[i]), dev.down(one[i])
            if M > 64 or layout == 0:
                assert np.array_equal(got, ref)
            else:
                assert max_rel_err(got, ref) < 1e-3
            if epi != dev.capi.EPI_BIAS_GELU:
                assert max_rel_err(ref, po.round_f16(po.gemm(X, np.ascontiguousarray(Ws[i].T), 1) + bs[i])) < 2e-3


@pytest.mark.parametrize("M", [5, 32])
def test_members_of_many_features_are_weight_streaming_launches_of_their_own(dev, po, stream, M):
    """Fragment blocks: three times 12288 features are more than one wave a feature tile can hold on the chip; one member is not."""
    N, K, layout = 12288, 1024, 2
    X, Ws, b = rnd(po, M * K, 81).reshape(M, K), [rnd(po, N * K, 82 + i, 0.05).reshape(N, K) for i in range(3)], rnd(po, N, 85, 0.3)
    dX, dB, dW = dev.up(X, 1), dev.up(b, 1), [weight(dev, W, layout) for W in Ws]
    one, three = [[dev.empty((M, N), 1) for _ in range(3)] for _ in range(2)]
    ptrs = lambda ts: (C.c_void_p * 3)(*[t.data_ptr() for t in ts])
    alone = [launches(dev, stream, "lg_gemm_fused_f16", layout, N, M, K, dW[i], K, dX, K, one[i], 1, dev.capi.EPI_BIAS_HEADS, dB, 1, 128, 0) for i in range(3)]
    got = launches(dev, stream, "lg_gemm_fused_grouped_f16", layout, N, M, K, 3, ptrs(dW), K, dX, K, ptrs(three), (C.c_int * 3)(1, 1, 1), dev.capi.EPI_BIAS_HEADS,
                   ptrs([dB] * 3), 1, 128, 0)
    assert [len(a) for a in alone] == [1, 1, 1] and got == alone[0] + alone[1] + alone[2]
    for i in range(3):
        assert np.array_equal(dev.down(one[i]), dev.down(three[i]))
    assert max_rel_err(dev.down(one[2]).reshape(M, N), po.round_f16(po.gemm(X, np.ascontiguousarray(Ws[2].T), 1) + b)) < 2e-3


def test_a_stream_can_be_made_known_while_one_is_captured(dev):
    """The set-up of a stream's workspace keeps off the null stream and out of captures: a (relaxed) capture that is open on a blocking
    stream goes on, with nothing in it, when a stream is created, when the stream that is captured is attached, and the null stream."""
    hip = dev.lib
    for case in ("create", "attach captured", "attach null"):
        s, graph, made, n = C.c_void_p(), C.c_void_p(), C.c_void_p(), C.c_size_t(7)
        dev.lib.lg_stream_detach(None)
        dev.sync()
        assert hip.hipStreamCreate(C.byref(s)) == 0 and hip.hipStreamBeginCapture(s, 2) == 0
        rc = dev.lib.lg_stream_create(C.byref(made)) if case == "create" else dev.lib.lg_stream_attach(s if case == "attach captured" else None, 0)
        assert hip.hipStreamEndCapture(s, C.byref(graph)) == 0 and rc == 0, dev.capi.last_error()
        assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0 and n.value == 0
        if made:
            assert dev.lib.lg_stream_destroy(made) == 0
        if case == "attach captured":
            assert dev.lib.lg_stream_detach(s) == 0
        assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(s) == 0
    assert dev.lib.lg_stream_attach(C.c_void_p(dev.stream), 0) == 0     # as the fixture left it


@pytest.mark.parametrize("M,N,K", [(11, 4096, 4096), (200, 4096, 4096), (256, 6144, 12288)])
def test_sliced_launches_replayed_between_eager_ones(dev, po, stream, M, N, K):
    """K-slices that meet in small tiles and in large ones: every replay, and the plain calls between them on the same workspace, end
    with the counters where they were and have the same bits."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    dX, dW = torch.randn(M, K, device="cuda", generator=gen).half(), (torch.randn(N * K, device="cuda", generator=gen) * 0.02).half()
    y, z = dev.empty((M, N), 1), dev.empty((M, N), 1)
    seen = []

    def between():
        assert dev.lib.lg_gemm_f16(2, 0, N, M, K, dW.data_ptr(), K, dX.data_ptr(), K, z.data_ptr(), N, stream) == 0
        dev.sync()
        seen.append((y.clone(), z.clone()))
        y.fill_(0.0)
        z.fill_(0.0)
        dev.sync()

    assert len(launches(dev, stream, "lg_gemm_f16", 2, 0, N, M, K, dW, K, dX, K, y, N, replays=4, between=between)) == 1
    assert all(torch.equal(a, seen[0][0]) and torch.equal(b, seen[0][0]) for a, b in seen) and bool(seen[0][0].any())


def test_a_group_whose_slices_do_not_fit_has_the_bits_of_its_members(dev, stream):
    """Members in two K-slices, three of which need more than the workspace: the group must not go to an unsliced kernel instead."""
    M, N, K = 256, 12288, 4096
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    dX = torch.randn(M, K, device="cuda", generator=gen).half()
    dW = [(torch.randn(N * K, device="cuda", generator=gen) * 0.02).half() for _ in range(3)]
    dB = torch.randn(N, device="cuda", generator=gen).half()
    one, three = [[dev.empty((M, N), 1) for _ in range(3)] for _ in range(2)]
    ptrs = lambda ts: (C.c_void_p * 3)(*[t.data_ptr() for t in ts])
    for i in range(3):
        launches(dev, stream, "lg_gemm_fused_f16", 0, N, M, K, dW[i], N, dX, K, one[i], N, dev.capi.EPI_BIAS, dB, 0, 0, 0)
    launches(dev, stream, "lg_gemm_fused_grouped_f16", 0, N, M, K, 3, ptrs(dW), N, dX, K, ptrs(three), (C.c_int * 3)(N, N, N), dev.capi.EPI_BIAS, ptrs([dB] * 3), 0, 0, 0)
    for i in range(3):
        assert torch.equal(one[i], three[i]) and bool(torch.isfinite(one[i]).all())
