"""GEMV launches captured in a HIP graph (torch.cuda.CUDAGraph) replay to the
same bits as the eager launches, replay after replay, with eager work and
input changes in between (the decode loop's use of the library)."""
from __future__ import annotations

import contextlib
import gc

import numpy as np
import pytest
import torch

import sllm_qmm as sq

from _helpers import make_raw, make_x

pytestmark = pytest.mark.gpu


def test_graph_replays_match_eager():
    torch.cuda.set_device(0)
    K = 1024
    specs = [("q4_1", 512), ("q4_1", 128), ("q4_1", 128), ("q8", 256), ("q5", 96), ("q5k1", 64)]
    ws = [sq.DeviceWeight.from_quant(sq.QuantWeight(q, make_raw(q, n, K, seed=i), K // 32, n, K))
          for i, (q, n) in enumerate(specs)]
    x = torch.from_numpy(make_x(1, K, seed=5)).cuda()
    outs = [torch.empty(w.rows, device="cuda") for w in ws]
    P = lambda t: t.data_ptr()

    def seq(stream):
        sq.matmul_multi_dev(ws[:3], P(x), 1, K, [P(o) for o in outs[:3]], stream)
        for w, o in zip(ws[3:], outs[3:]):
            sq.matmul_dev(w, P(x), 1, K, P(o), stream)

    def eager():
        seq(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return [o.clone() for o in outs]

    want = eager()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        seq(torch.cuda.current_stream().cuda_stream)
    for rep in range(4):
        for o in outs:
            o.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        for i, (o, w) in enumerate(zip(outs, want)):
            assert torch.equal(o.view(torch.int32), w.view(torch.int32)), f"replay {rep}, weight {i}"
        eager()  # eager work between replays

    # the graph reads x's current contents: new input, same as eager on it
    x.copy_(torch.from_numpy(make_x(1, K, seed=6)).cuda())
    want2 = eager()
    assert not torch.equal(want2[0], want[0])
    g.replay()
    torch.cuda.synchronize()
    for o, w in zip(outs, want2):
        assert torch.equal(o.view(torch.int32), w.view(torch.int32))


def test_workspace_growth_keeps_captured_graphs_valid():
    # A decode step captured on a stream (its attention keeps the rotated q
    # rows in the stream's workspace), then a large prefill on the same
    # stream grows that workspace: the old buffer must stay valid, so the
    # graph still replays to the eager result.
    from test_gpu_attention import Model
    from sllm_qmm import synth
    rng = np.random.default_rng(3)
    H, KV, DK, K = 8, 2, 128, 1024
    m = Model(H, KV, DK, 64, rng, base=500000.0)
    kv = sq.KVCache(1, KV, DK, 256)
    kv.set_length(100)
    q = torch.from_numpy(rng.normal(size=H * DK).astype(np.float32)).cuda()
    k = torch.from_numpy(rng.normal(size=KV * DK).astype(np.float32)).cuda()
    v = torch.from_numpy(rng.normal(size=KV * DK).astype(np.float32)).cuda()
    att = torch.empty(H * DK, device="cuda")
    w = sq.DeviceWeight.from_quant(sq.QuantWeight("q4_1", make_raw("q4_1", 512, K, seed=1), K // 32, 512, K))
    y = torch.empty(512, device="cuda")
    P = lambda t: t.data_ptr()
    s = torch.cuda.Stream()

    def step(sp):
        kv.set_length(100)
        sq.attention_dev(kv, 0, m.params, P(q), P(k), P(v), 1, 100, P(att), sp)
        sq.matmul_dev(w, P(att), 1, K, P(y), sp)

    with torch.cuda.stream(s):
        step(s.cuda_stream)  # eager: the workspace is allocated here, before the capture
    s.synchronize()
    want = (att.clone(), y.clone())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        step(s.cuda_stream)
    # prefill on the same stream: M = 512, K = 14336 needs far more workspace
    F = 14336
    big = sq.load_weight_f32_direct(synth.GGML_Q4_K, synth.q4k_blocks(5, 256, F), 256, F)
    xb = torch.from_numpy(make_x(512, F, seed=2)).cuda()
    yb = torch.empty(512 * 256, device="cuda")
    with torch.cuda.stream(s):
        sq.matmul_dev(big, P(xb), 512, F, P(yb), s.cuda_stream)
    s.synchronize()
    for rep in range(3):
        att.fill_(float("nan"))
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(att.view(torch.int32), want[0].view(torch.int32)), rep
        assert torch.equal(y.view(torch.int32), want[1].view(torch.int32)), rep
        with torch.cuda.stream(s):
            sq.matmul_dev(big, P(xb), 512, F, P(yb), s.cuda_stream)  # eager work in between
        s.synchronize()
    kv.close()


def test_workspace_growth_under_capture_is_an_error_and_reserve_avoids_it():
    from sllm_qmm import synth
    F, M = 8192, 256
    big = sq.load_weight_f32_direct(synth.GGML_Q4_K, synth.q4k_blocks(6, 128, F), 128, F)
    xb = torch.from_numpy(make_x(M, F, seed=3)).cuda()
    yb = torch.empty(M * 128, device="cuda")
    small = sq.DeviceWeight.from_quant(sq.QuantWeight("q8", make_raw("q8", 64, 256, seed=2), 8, 64, 256))
    xs = torch.from_numpy(make_x(1, 256, seed=4)).cuda()
    ys = torch.empty(64, device="cuda")
    P = lambda t: t.data_ptr()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    err = None
    with torch.cuda.graph(g, stream=s):
        sq.matmul_dev(small, P(xs), 1, 256, P(ys), s.cuda_stream)  # no workspace
        try:
            sq.matmul_dev(big, P(xb), M, F, P(yb), s.cuda_stream)  # would allocate: refused
        except sq.SllmError as e:
            err = e
    assert err is not None and err.status == 1 and "sllm_workspace_reserve" in str(err)
    del g
    # reserved before the capture, the same call captures and replays to the eager result
    s2 = torch.cuda.Stream()
    sq.workspace_reserve(s2.cuda_stream, 64 << 20)
    with torch.cuda.stream(s2):
        sq.matmul_dev(big, P(xb), M, F, P(yb), s2.cuda_stream)
    s2.synchronize()
    want = yb.clone()
    g2 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g2, stream=s2):
        sq.matmul_dev(big, P(xb), M, F, P(yb), s2.cuda_stream)
    for rep in range(3):
        yb.fill_(float("nan"))
        g2.replay()
        torch.cuda.synchronize()
        assert torch.equal(yb.view(torch.int32), want.view(torch.int32)), rep


@contextlib.contextmanager
def _capture(g, stream):
    # no garbage collection inside: it could destroy an earlier graph or weight, which
    # synchronizes the device, while this one is being captured
    gc.collect()
    gc.disable()
    try:
        with torch.cuda.graph(g, stream=stream):
            yield
    finally:
        gc.enable()


def _captured(call, stream):
    g = torch.cuda.CUDAGraph()
    with _capture(g, stream):
        call(stream.cuda_stream)
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
    return g


def _matmul(w, x, stream=0):
    y = torch.full((x.shape[0], w.rows), float("nan"), device="cuda")
    sq.matmul_dev(w, x.data_ptr(), x.shape[0], x.shape[1], y.data_ptr(), stream)
    return y


@pytest.mark.parametrize("qtype,N,K,M", [("q5", 96, 512, 15), ("q4_1", 40, 4096, 6), ("q8", 96, 512, 15),
                                         ("q5k1", 4097, 256, 5)])
def test_capture_without_workspace_takes_the_gemv_below_the_tiled_gemms_rows(qtype, N, K, M):
    w = sq.DeviceWeight.from_quant(sq.QuantWeight(qtype, make_raw(qtype, N, K, seed=1), K // 32, N, K))
    x = torch.from_numpy(make_x(M, K, seed=2)).cuda()
    eager = _matmul(w, x)
    sq.set_param("gemm_min_rows", 1 << 20)
    gemv = _matmul(w, x)
    sq.set_param("gemm_min_rows", 0)
    y = torch.empty_like(gemv)
    g = _captured(lambda s: sq.matmul_dev(w, x.data_ptr(), M, K, y.data_ptr(), s), torch.cuda.Stream())
    assert torch.equal(y, gemv) and not torch.equal(y, eager)
    del g


@pytest.mark.parametrize("qtype,N,K,M", [("q5", 96, 512, 16), ("q5", 96, 512, 300), ("q8", 96, 512, 16),
                                         ("q4_1", 40, 4096, 33)])
def test_capture_without_workspace_refuses_the_tiled_gemms_rows(qtype, N, K, M):
    w = sq.DeviceWeight.from_quant(sq.QuantWeight(qtype, make_raw(qtype, N, K, seed=1), K // 32, N, K))
    x = torch.from_numpy(make_x(M, K, seed=2)).cuda()
    y = torch.zeros((M, N), device="cuda")
    s, err = torch.cuda.Stream(), None
    g = torch.cuda.CUDAGraph()
    with _capture(g, s):
        y.fill_(1.0)
        try:
            sq.matmul_dev(w, x.data_ptr(), M, K, y.data_ptr(), s.cuda_stream)
        except sq.SllmError as e:
            err = (e.status, str(e))
    del g
    assert err is not None and err[0] == 1 and "sllm_workspace_reserve" in err[1]


def test_capture_decides_for_each_weight_by_itself():
    # the workspace holds the small weight's GEMM, not the large one's: beside it the
    # small weight still gives its single call's bits
    from test_gpu_kquant_native import make_kq
    K, M = 2048, 9
    small, large = (sq.load_weight_f32_direct(10, make_kq(10, n, K, n), n, K) for n in (96, 8192))
    x = torch.from_numpy(make_x(M, K, seed=3)).cuda()
    sq.set_param("gemm_splits", 16)  # 16 x 9 x 8192 floats of partial sums: more than the 4 MiB a stream starts with
    try:
        sq.set_param("gemm_min_rows", 1 << 20)
        gemv = [_matmul(w, x) for w in (small, large)]
        sq.set_param("gemm_min_rows", 0)
        single = _matmul(small, x)
        s = torch.cuda.Stream()
        sq.workspace_reserve(s.cuda_stream, 1)
        ys = [torch.empty_like(t) for t in gemv]
        nys = [torch.empty_like(t) for t in gemv]
        ones = torch.ones(K, device="cuda")

        def call(st):
            sq.matmul_multi_dev([small, large], x.data_ptr(), M, K, [y.data_ptr() for y in ys], st)
            sq.rmsnorm_matmul_multi_dev([small, large], x.data_ptr(), ones.data_ptr(), 1e-5, M, K,
                                        [y.data_ptr() for y in nys], st)
        g = _captured(call, s)
    finally:
        sq.set_param("gemm_splits", 0)
        sq.set_param("gemm_min_rows", 0)
    assert not torch.equal(single, gemv[0])
    assert torch.equal(ys[0], single) and torch.equal(ys[1], gemv[1])
    assert all(torch.isfinite(y).all() for y in nys)
    del g


@pytest.mark.parametrize("M", [6, 12])
def test_capture_of_a_mixed_gate_up_pair_without_workspace(M):
    # int8 weights of two formats: the pair needs buffers of its own, so a stream
    # without workspace refuses; with a little reserved it runs
    K, N = 4096, 64
    ws = [sq.DeviceWeight.from_quant(sq.QuantWeight(q, make_raw(q, N, K, seed=5), K // 32, N, K)) for q in ("q8", "q4_1")]
    x = torch.from_numpy(make_x(M, K, seed=6)).cuda()
    nw = torch.ones(K, device="cuda")
    h, want = (torch.full((M, N), float("nan"), device="cuda") for _ in range(2))
    call = lambda y: lambda s: sq.rmsnorm_matmul_swiglu_dev(*ws, x.data_ptr(), nw.data_ptr(), 1e-5, M, K, y.data_ptr(), s)
    call(want)(0)
    s = torch.cuda.Stream()
    sq.workspace_reserve(s.cuda_stream, 1)
    g = _captured(call(h), s)
    assert torch.isfinite(want).all() and torch.equal(h, want)
    del g
