"""GPU tests of the prefill GEMM of the native Q2_K / Q3_K weights (bf16 matrix
cores over the exact three-way split of the fp32 activations).

Bound: a weight is dl * q - ml. The GEMM forms every product of q and of ml
exactly or with one rounding and adds them in some order, the oracle multiplies
the rounded weights and adds sequentially: both are within (K + K / 32 + 64) u
of sum |x| (|dl q| + |ml|), u = 2^-24.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
import sllm_qmm as sq

from _helpers import make_x
from test_gpu_kquant_native import PER, make_kq

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


@pytest.fixture(autouse=True)
def _params():
    sq.set_param("gemm_min_rows", 1)
    yield
    for p in ("gemm_min_rows", "gemm_shape", "gemm_splits"):
        sq.set_param(p, 0)


def parts(t, raw, N, K):
    """|dl q| + |ml| of every weight."""
    a = raw.reshape(-1, PER[t]).copy()
    if t == 11:
        return np.abs(oracle.dense_weights(t, raw, N, K)).astype(np.float64)
    b = a.copy()
    a[:, 82:84] = 0
    b[:, 80:82] = 0
    return sum(np.abs(oracle.dense_weights(t, r.reshape(-1), N, K)).astype(np.float64) for r in (a, b))


def gemm(w, x):
    M, K = x.shape
    xd = torch.from_numpy(x).cuda()
    y = torch.full((M, w.rows), float("nan"), device="cuda")
    sq.matmul_dev(w, xd.data_ptr(), M, K, y.data_ptr())
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("t", [10, 11])
@pytest.mark.parametrize("N,K,M,shape,splits", [
    (1, 256, 1, 0, 0), (300, 768, 32, 0, 0), (300, 768, 33, 0, 0), (257, 512, 65, 0, 0), (31, 256, 129, 0, 0),
    (513, 1280, 200, 0, 0), (520, 1024, 100, 1, 3), (520, 1024, 100, 2, 5), (520, 1024, 100, 3, 2),
    (256, 2048, 4, 0, 32)])
def test_gemm_within_bound(t, N, K, M, shape, splits):
    sq.set_param("gemm_shape", shape)
    sq.set_param("gemm_splits", splits)
    raw = make_kq(t, N, K, 31 + M)
    w = sq.load_weight_f32_direct(t, raw, N, K)
    x = make_x(M, K, seed=M)
    ref = oracle.matmul_dense(oracle.dense_weights(t, raw, N, K), x).astype(np.float64)
    bound = (K + K // 32 + 64) * U * (np.abs(x).astype(np.float64) @ parts(t, raw, N, K).T) + 1e-30
    assert np.all(np.abs(gemm(w, x) - ref) <= bound)


@pytest.mark.parametrize("t", [10, 11])
def test_activations_outside_the_factored_range(t):
    # huge, tiny, infinite and NaN activations in single rows and blocks: the
    # blocks that hold one are computed weight by weight, as the reference does
    N, K, M = 70, 512, 40
    raw = make_kq(t, N, K, 5)
    w = sq.load_weight_f32_direct(t, raw, N, K)
    W = oracle.dense_weights(t, raw, N, K)
    x = make_x(M, K, seed=6)
    x[3] *= np.float32(2.0 ** 100)
    x[7] *= np.float32(2.0 ** -110)
    x[11, 64:96] = np.float32(3e38)
    x[35, 5] = np.inf
    x[36, 300] = -np.inf
    x[37, 511] = np.nan
    got = gemm(w, x).astype(np.float64)
    with np.errstate(over="ignore", invalid="ignore"):
        ref = oracle.matmul_dense(W, x).astype(np.float64)
        bound = (K + K // 32 + 64) * U * (np.abs(x).astype(np.float64) @ parts(t, raw, N, K).T) + 1e-44
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf])
    fin = np.isfinite(ref)
    assert np.all(np.abs(got[fin] - ref[fin]) <= bound[fin])


@pytest.mark.parametrize("t", [10, 11])
def test_weights_with_infinite_scales_stay_on_the_gemv(t):
    # inf * 0 per weight is NaN, inf * (a group's sum) is not: such a weight
    # gives the same bits whether the GEMM is allowed or not
    N, K, M = 40, 512, 9
    raw = make_kq(t, N, K, 8).reshape(-1, PER[t])
    at = 80 if t == 10 else 108
    raw[5, at:at + 2] = [0x00, 0x7C]
    if t == 10:
        raw[9, 82:84] = [0x00, 0xFC]
    w = sq.load_weight_f32_direct(t, raw.reshape(-1), N, K)
    x = make_x(M, K, seed=9)
    a = gemm(w, x)
    sq.set_param("gemm_min_rows", 1 << 20)
    assert np.array_equal(a.view(np.uint32), gemm(w, x).view(np.uint32))


@pytest.mark.parametrize("t", [10, 11])
def test_capture_without_workspace_takes_the_gemv(t):
    # the GEMV needs no workspace: a stream under capture that has none records
    # it, and the replays equal the eager GEMV bit for bit
    N, K, M = 96, 512, 9
    w = sq.load_weight_f32_direct(t, make_kq(t, N, K, 12), N, K)
    x = torch.from_numpy(make_x(M, K, seed=13)).cuda()
    y = torch.empty((M, N), device="cuda")
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        sq.matmul_dev(w, x.data_ptr(), M, K, y.data_ptr(), s.cuda_stream)
    sq.set_param("gemm_min_rows", 1 << 20)
    want = gemm(w, x.cpu().numpy())
    for _ in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy().view(np.uint32), want.view(np.uint32))


def test_q2k_weights_that_nearly_cancel():
    # dl q and ml close together: rows of exact zeros give exact zeros, and the error
    # is in |w| (dl (q - b) and w_b are within 3 |w|), not in |dl q| + |ml|
    N, K, M = 96, 1024, 48
    rng = np.random.default_rng(21)
    raw = make_kq(10, N, K, 22).reshape(N, K // 256, 84)
    code = (np.arange(N) % 3 + 1).astype(np.uint8)  # every code of a row
    sc = rng.integers(1, 6, (N, K // 256, 16)).astype(np.uint8)
    raw[..., :16] = sc | ((sc * code[:, None, None]) << 4)
    raw[..., 16:80] = (code * 0x55)[:, None, None]
    d = np.float16(2.0 ** -6)
    dm = np.full(N, d)
    dm[N // 2:] = np.float16(2.0 ** -6 * (1 + 2.0 ** -9))
    raw[..., 80:82] = np.frombuffer(d.tobytes(), np.uint8)
    raw[..., 82:84] = dm.view(np.uint8).reshape(N, 1, 2)
    raw = raw.reshape(-1)
    W = oracle.dense_weights(10, raw, N, K)
    assert not W[:N // 2].any() and W[N // 2:].all()
    w = sq.load_weight_f32_direct(10, raw, N, K)
    x = make_x(M, K, seed=23)
    got = gemm(w, x)
    assert not got[:, :N // 2].any()
    ref = oracle.matmul_dense(W, x).astype(np.float64)
    bound = 3 * (K + K // 32 + 64) * U * (np.abs(x).astype(np.float64) @ np.abs(W).T.astype(np.float64))
    assert np.all(np.abs(got - ref) <= bound)


@pytest.mark.parametrize("t", [10, 11])
@pytest.mark.parametrize("N,K,M,gemm_from", [(512, 2048, 8, 9), (512, 2048, 9, 9), (64, 4096, 6, 7), (64, 4096, 7, 7),
                                             (4096, 1024, 6, 7), (4096, 1024, 7, 7)])
def test_the_line_between_gemv_and_gemm(t, N, K, M, gemm_from):
    w = sq.load_weight_f32_direct(t, make_kq(t, N, K, 41), N, K)
    x = make_x(M, K, seed=42)
    forced = gemm(w, x)
    sq.set_param("gemm_min_rows", 1 << 20)
    gemv = gemm(w, x)
    sq.set_param("gemm_min_rows", 0)
    assert not np.array_equal(gemv, forced)  # two orders
    assert np.array_equal(gemm(w, x), forced if M >= gemm_from else gemv)


@pytest.mark.parametrize("t", [10, 11])
@pytest.mark.parametrize("K,M", [(4096, 8), (14336, 8), (14336, 33), (4096, 130)])
def test_gemm_is_as_close_to_64_bits_as_the_gemv(t, K, M):
    # many K splits included (these shapes take up to 32): their sums are added in
    # trees, not in one chain
    N = 256
    raw = make_kq(t, N, K, 51)
    w = sq.load_weight_f32_direct(t, raw, N, K)
    x = np.random.default_rng(52).normal(size=(M, K)).astype(np.float32)
    ref = x.astype(np.float64) @ oracle.dense_weights(t, raw, N, K).astype(np.float64).T
    err = lambda y: np.linalg.norm(y - ref) / np.linalg.norm(ref)
    e = err(gemm(w, x))
    sq.set_param("gemm_min_rows", 1 << 20)
    assert e <= 1.03 * err(gemm(w, x))
