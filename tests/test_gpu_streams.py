"""Kernel-layer calls that use the library's scratch, on several streams at once and
under capture: each result has the bits of the same call made alone."""
import ctypes

import numpy as np
import pytest
import torch

import uaii_amd
from uaii_amd import synth, DeviceWeight, check_hip

pytestmark = pytest.mark.gpu

I64 = ctypes.c_int64


def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def raw(stream):
    return ctypes.c_void_p(stream.cuda_stream)


def weight(t, rows, cols, seed):
    return DeviceWeight(t, synth.quantize(t, synth.normals(seed, 1, 0, rows * cols, 0.02)), rows, cols)


def rows_of(m, cols, seed):
    return torch.from_numpy(synth.normals(seed, 2, 0, m * cols, 1.0).reshape(m, cols)).cuda()


@pytest.mark.parametrize("t", [uaii_amd.Q5_K, uaii_amd.Q4_0, uaii_amd.F16], ids=lambda t: uaii_amd.TYPE_NAMES[t])
@pytest.mark.parametrize("m", [9, 300])  # split over K with its partials, and not
def test_row_products_on_streams(hip, t, m):
    """Six streams, more than there are kept buffers, and the null stream."""
    rows, cols, n = 1024, 2048, 6
    w = weight(t, rows, cols, 3)
    xs = [rows_of(m, cols, 10 + i) for i in range(n)]
    want = []
    for x in xs:
        y = torch.zeros(m, rows, device="cuda")
        check_hip(hip.uaii_hip_gemm(w.h, ptr(x), I64(m), ptr(y), None))
        torch.cuda.synchronize()
        want.append(y)
    streams = [torch.cuda.Stream() for _ in range(n)]
    ys = [torch.zeros(8, m, rows, device="cuda") for _ in range(n)]
    y0 = torch.zeros(8, m, rows, device="cuda")
    torch.cuda.synchronize()
    for k in range(8):
        for i in range(n):
            check_hip(hip.uaii_hip_gemm(w.h, ptr(xs[i]), I64(m), ptr(ys[i][k]), raw(streams[i])))
        check_hip(hip.uaii_hip_gemm(w.h, ptr(xs[0]), I64(m), ptr(y0[k]), None))
    torch.cuda.synchronize()
    for k in range(8):
        assert torch.equal(y0[k], want[0])
        for i in range(n):
            assert torch.equal(ys[i][k], want[i]), (i, k)


def test_attention_beside_row_product(hip):
    """Decode attention on one stream, a row product on another."""
    nh, nkv, hd, seq = 8, 4, 64, 1024
    g = torch.Generator().manual_seed(1)
    q = torch.randn(nh * hd, generator=g).cuda()
    k, v = (torch.randn(nkv, seq, hd, generator=g).half().cuda() for _ in range(2))
    m, cols, rows = 64, 2048, 512
    w, x = weight(uaii_amd.Q5_K, rows, cols, 5), rows_of(m, cols, 6)

    def attend(out, s):
        check_hip(hip.uaii_hip_attention_decode(ptr(q), ptr(k), ptr(v), 1, I64(seq), nh, nkv, hd, I64(1000), ptr(out), s))

    def product(y, s):
        check_hip(hip.uaii_hip_gemm(w.h, ptr(x), I64(m), ptr(y), s))

    o0, y0 = torch.zeros(nh * hd, device="cuda"), torch.zeros(m, rows, device="cuda")
    attend(o0, None)
    torch.cuda.synchronize()
    product(y0, None)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    os_, ys = torch.zeros(16, nh * hd, device="cuda"), torch.zeros(16, m, rows, device="cuda")
    torch.cuda.synchronize()
    for i in range(16):
        attend(os_[i], raw(a))
        product(ys[i], raw(b))
    torch.cuda.synchronize()
    for i in range(16):
        assert torch.equal(os_[i], o0) and torch.equal(ys[i], y0), i


@pytest.mark.parametrize("t", [uaii_amd.Q5_K, uaii_amd.F16, uaii_amd.Q4_0, uaii_amd.Q6_K],
                         ids=lambda t: uaii_amd.TYPE_NAMES[t])
def test_captured_row_product(hip, t):
    """A captured call replayed on new inputs after larger calls, eager and captured,
    made the library grow what it keeps. Captured Q5_K and F16 calls are the per-row
    kernel's bits; the others those of the eager call."""
    m, rows, cols = 9, 512, 1024
    w = weight(t, rows, cols, 7)
    x, y = rows_of(m, cols, 20), torch.zeros(m, rows, device="cuda")
    s = torch.cuda.Stream()

    def capture(m, x, y, w):
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            check_hip(hip.uaii_hip_gemm(w.h, ptr(x), I64(m), ptr(y), raw(s)))
        return graph

    graph = capture(m, x, y, w)
    big_m, big = 700, weight(t, 2048, 2048, 8)
    bx, by, bz = rows_of(big_m, 2048, 9), *(torch.zeros(big_m, 2048, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    for stream in (raw(s), None):
        check_hip(hip.uaii_hip_gemm(big.h, ptr(bx), I64(big_m), ptr(by), stream))
    big_graph = capture(big_m, bx, bz, big)
    big_graph.replay()
    torch.cuda.synchronize()
    if t in (uaii_amd.Q4_0, uaii_amd.Q6_K):
        assert torch.equal(by, bz)
    for i in range(4):
        x.copy_(rows_of(m, cols, 30 + i))
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = torch.zeros(m, rows, device="cuda")
        if t in (uaii_amd.Q5_K, uaii_amd.F16):
            for r in range(m):
                check_hip(hip.uaii_hip_gemv(w.h, ptr(x[r]), ptr(want[r]), None))
        else:
            check_hip(hip.uaii_hip_gemm(w.h, ptr(x), I64(m), ptr(want), None))
        torch.cuda.synchronize()
        assert torch.equal(y, want), i
