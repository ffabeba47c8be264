"""GPU tests of the short-prompt GEMM (int8 formats, up to 32 activation rows):
edges of its 32 x 32 tiles, of the K split over a workgroup's waves
(fewer, as many and more chunks than waves), shared-input launches, the residual
add, the SwiGLU epilogue and the fused norm. Bound: 1e-5 of sum |terms|, as for
the tiled GEMM (its rounding is the same, its order another)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
import sllm_qmm as sq

from _helpers import REL_TOL, make_raw, make_x, term_abs_sum

pytestmark = pytest.mark.gpu
QTYPES = ["q8", "q4", "q4_1", "q5k1"]


@pytest.fixture(autouse=True)
def _params():
    sq.set_param("gemm_min_rows", 1)
    yield
    sq.set_param("gemm_min_rows", 0)


def weight(qtype, N, K, seed):
    raw = make_raw(qtype, N, K, seed=seed)
    return raw, sq.DeviceWeight.from_quant(sq.QuantWeight(qtype, raw, K // 32, N, K))


def run(w, x):
    M, K = x.shape
    xd = torch.from_numpy(x).cuda()
    y = torch.full((M, w.rows), float("nan"), device="cuda")
    sq.matmul_dev(w, xd.data_ptr(), M, K, y.data_ptr())
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("qtype", QTYPES)
@pytest.mark.parametrize("N,K,M", [(1, 256, 1), (31, 256, 7), (33, 512, 32), (2100, 2304, 31), (2048, 8192, 5),
                                   (257, 2048, 16), (8230, 256, 3), (96, 1792, 2)])
def test_against_the_oracle(qtype, N, K, M):
    raw, w = weight(qtype, N, K, N + M)
    x = make_x(M, K, seed=K + M)
    err = np.abs(run(w, x).astype(np.float64) - oracle.matmul(qtype, raw, N, x))
    assert np.all(err <= REL_TOL * term_abs_sum(qtype, raw, N, x) + 1e-30)


def test_q5k_weights_in_one_and_two_mfmas():
    from sllm_qmm import synth
    N, K, M = 70, 1024, 30
    raw = synth.q5k_blocks(3, N, K)
    w = sq.load_weight_f32_direct(synth.GGML_Q5_K, raw, N, K)
    assert w.q5k1_one_mfma
    qt, ref = oracle.load_weight(synth.GGML_Q5_K, raw, N, K)
    x = make_x(M, K, seed=4)
    err = np.abs(run(w, x).astype(np.float64) - oracle.matmul(qt, ref, N, x))
    assert np.all(err <= REL_TOL * term_abs_sum(qt, ref, N, x) + 1e-30)


@pytest.mark.parametrize("M,K", [(3, 1024), (32, 1024), (5, 2304), (16, 4096), (30, 8192)])
def test_shared_input_add_swiglu_and_norm_equal_the_single_calls(M, K):
    # bit for bit: an output's order depends on K alone, not on the launch (alone, a
    # weight this narrow is cut into K splits above 2048 columns)
    _, a = weight("q4_1", 300, K, 1)
    _, b = weight("q8", 65, K, 2)
    _, c = weight("q4_1", 300, K, 3)
    ws = [a, b, c]
    x = make_x(M, K, seed=5)
    single = [run(w, x) for w in ws]
    xd = torch.from_numpy(x).cuda()
    outs = [torch.full((M, w.rows), float("nan"), device="cuda") for w in ws]
    sq.matmul_multi_dev(ws, xd.data_ptr(), M, K, [o.data_ptr() for o in outs])
    h, g, u = (torch.full((M, 300), float("nan"), device="cuda") for _ in range(3))
    sq.matmul_swiglu_dev(a, c, xd.data_ptr(), M, K, h.data_ptr(), g.data_ptr(), u.data_ptr())
    base = np.random.default_rng(6).normal(size=(M, 300)).astype(np.float32)
    dst = torch.from_numpy(base).cuda()
    sq.matmul_add_dev(a, xd.data_ptr(), M, K, dst.data_ptr())
    nw = np.random.default_rng(7).normal(1, 0.2, K).astype(np.float32)
    nwd = torch.from_numpy(nw).cuda()
    nouts = [torch.full((M, w.rows), float("nan"), device="cuda") for w in ws]
    sq.rmsnorm_matmul_multi_dev(ws, xd.data_ptr(), nwd.data_ptr(), 1e-5, M, K, [o.data_ptr() for o in nouts])
    torch.cuda.synchronize()
    bits = lambda t: (t.cpu().numpy() if isinstance(t, torch.Tensor) else t).view(np.uint32)
    for o, s in zip(outs, single):
        assert np.array_equal(bits(o), bits(s))
    assert np.array_equal(bits(dst), bits(base + single[0]))
    for o, s in ((g, single[0]), (u, single[2])):
        assert np.array_equal(bits(o), bits(s))
    want = oracle.swiglu(g.cpu().numpy(), u.cpu().numpy())
    assert np.all(np.abs(h.cpu().numpy() - want) <= 2.0 ** -21 * np.abs(want) + 1e-30)
    normed = np.stack([oracle.rmsnorm(x[i:i + 1], nw, 1e-5, lib_order=True)[0] for i in range(M)])
    for o, w in zip(nouts, ws):
        assert np.array_equal(bits(o), bits(run(w, normed)))


@pytest.mark.parametrize("qtype", QTYPES)
def test_nonfinite_scales_and_huge_activations_follow_the_reference(qtype):
    # chunks with such a scale are computed in the reference's operation order
    N, K, M = 40, 2048, 9
    raw, _ = weight(qtype, N, K, 8)
    raw = raw.copy()
    per = {"q8": 34, "q4": 18, "q4_1": 20, "q5k1": 20}[qtype]
    blocks = raw.reshape(-1, per)
    for i, bits in ((5, 0x7C00), (70, 0xFC00), (400, 0x7E00)):
        blocks[i, 0:2] = [bits & 0xFF, bits >> 8]
    w = sq.DeviceWeight.from_quant(sq.QuantWeight(qtype, raw, K // 32, N, K))
    x = make_x(M, K, seed=9)
    x[2, 300:400] *= np.float32(2.0 ** 98)
    got = run(w, x)
    with np.errstate(over="ignore", invalid="ignore"):
        ref = oracle.matmul(qtype, raw, N, x)
        bound = REL_TOL * term_abs_sum(qtype, raw, N, x)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert inf.any() and np.array_equal(got[inf], ref[inf])
    fin = np.isfinite(ref) & np.isfinite(bound)
    assert np.all(np.abs(got[fin].astype(np.float64) - ref[fin]) <= bound[fin])


@pytest.mark.parametrize("K", [768, 2304])
@pytest.mark.parametrize("qtype", QTYPES)
def test_wide_launches_equal_the_narrow_ones(qtype, K):
    # more tiles than CUs (four waves to a tile, two or four parts of K each, in a
    # gate / up pair four) against the same rows in a small weight's launch
    N, M = 8224, 7
    raw, w = weight(qtype, N, K, 11)
    n = 40
    per = raw.size // N
    x = make_x(M, K, seed=12)
    full = run(w, x)
    if qtype != "q5k1":  # (its raw form is two halves, each of all rows)
        small = sq.DeviceWeight.from_quant(sq.QuantWeight(qtype, raw[:n * per].copy(), K // 32, n, K))
        assert np.array_equal(full[:, :n].copy().view(np.uint32), run(small, x).view(np.uint32))
    xd = torch.from_numpy(x).cuda()
    h, g, u = (torch.full((M, N), float("nan"), device="cuda") for _ in range(3))
    sq.matmul_swiglu_dev(w, w, xd.data_ptr(), M, K, h.data_ptr(), g.data_ptr(), u.data_ptr())
    torch.cuda.synchronize()
    for o in (g, u):
        assert np.array_equal(o.cpu().numpy().view(np.uint32), full.view(np.uint32))


@pytest.mark.parametrize("qtype", ["q4_1", "q5k1"])
@pytest.mark.parametrize("N,K,M,gemm", [
    (4097, 256, 4, False), (4097, 256, 5, True), (4096, 256, 6, False), (4096, 256, 7, True), (40, 4096, 5, False),
    (40, 4096, 6, True), (40, 3840, 6, False), (40, 3840, 7, True), (40, 4352, 7, False), (4097, 4352, 7, False), (4097, 4352, 8, True)])
def test_the_line_between_gemv_and_short_prompt_gemm(qtype, N, K, M, gemm):
    _, w = weight(qtype, N, K, 13)
    x = make_x(M, K, seed=14)
    sq.set_param("gemm_min_rows", 1 << 20)
    gemv = run(w, x)
    sq.set_param("gemm_min_rows", 0)
    assert np.array_equal(run(w, x).view(np.uint32), gemv.view(np.uint32)) is not gemm


def _power_of_two_weight(qtype, N, K, rng):
    """Blocks whose scales are powers of two and mins small multiples of them, and
    the weights they stand for."""
    G = K // 32
    d = 2.0 ** rng.integers(-4, 1, (N, G))
    f16 = lambda v: v.astype(np.float16).view(np.uint8).reshape(N, G, 2)
    if qtype == "q8":
        q = rng.integers(-127, 128, (N, G, 32)).astype(np.int8)
        return np.concatenate([f16(d), q.view(np.uint8)], -1), (d[..., None] * q)
    q = rng.integers(0, 16, (N, G, 32)).astype(np.uint8)
    packed = q[..., :16] | (q[..., 16:] << 4)
    if qtype == "q4":
        return np.concatenate([f16(d), packed], -1), d[..., None] * (q.astype(np.int64) - 8)
    m = d * rng.integers(-8, 9, (N, G))
    lo = np.concatenate([f16(d), f16(m), packed], -1)
    w = d[..., None] * q + m[..., None]
    if qtype == "q4_1":
        return lo, w
    hb = rng.integers(0, 2, (N, G, 32)).astype(np.uint8)
    hi = np.concatenate([f16(16 * d), f16(0 * d), hb[..., :16] | (hb[..., 16:] << 4)], -1)
    return np.concatenate([lo.reshape(-1), hi.reshape(-1)]), w + 16 * d[..., None] * hb


@pytest.mark.parametrize("qtype", QTYPES)
@pytest.mark.parametrize("N,K,M", [(70, 512, 32), (33, 4096, 5), (4100, 768, 9)])
def test_exact_sums_equal_the_integer_result(qtype, N, K, M):
    # rows whose largest magnitude is 127 * 2^e quantize exactly (scale 2^e), block
    # scales are powers of two: every dot, term and sum fits 24 bits, so the outputs
    # pin the integer dots bit for bit
    rng = np.random.default_rng(N + K)
    raw, W = _power_of_two_weight(qtype, N, K, rng)
    w = sq.DeviceWeight.from_quant(sq.QuantWeight(qtype, np.ascontiguousarray(raw).reshape(-1), K // 32, N, K))
    x = np.zeros((M, K // 32, 32), np.float32)
    for i in range(M):  # a few blocks of each row hold values: sums stay small
        at = rng.choice(K // 32, 4, replace=False)
        v = rng.integers(-2, 3, (4, 32)).astype(np.float32)
        v[:, rng.integers(0, 32)] = 127
        x[i, at] = v * 2.0 ** (i % 3)
    x = x.reshape(M, K)
    want = x.astype(np.float64) @ W.reshape(N, K).T
    assert np.array_equal(run(w, x), want.astype(np.float32))


@pytest.mark.parametrize("M,K", [(5, 1024), (32, 1024), (9, 2304), (32, 4096)])
@pytest.mark.parametrize("qtype", QTYPES)
def test_normed_gate_up_pair_equals_norm_then_pair(qtype, M, K):
    _, a = weight(qtype, 97, K, 15)
    _, b = weight(qtype, 97, K, 16)
    x = make_x(M, K, seed=17)
    nw = np.random.default_rng(18).normal(1, 0.2, K).astype(np.float32)
    normed = np.stack([oracle.rmsnorm(x[i:i + 1], nw, 1e-5, lib_order=True)[0] for i in range(M)])
    xd, nd, wd = (torch.from_numpy(v).cuda() for v in (x, normed, nw))
    h, want = (torch.full((M, 97), float("nan"), device="cuda") for _ in range(2))
    sq.rmsnorm_matmul_swiglu_dev(a, b, xd.data_ptr(), wd.data_ptr(), 1e-5, M, K, h.data_ptr())
    sq.matmul_swiglu_dev(a, b, nd.data_ptr(), M, K, want.data_ptr())
    torch.cuda.synchronize()
    assert torch.isfinite(want).all() and torch.equal(h.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("over", ["gate", "up"])
@pytest.mark.parametrize("M", [9, 33])
def test_h_over_gate_or_up_holds_the_swiglu(M, over):
    # the same buffer for h and gate (or up): the tiled GEMM's pass leaves h there, and
    # so does the short-prompt GEMM's epilogue
    _, a = weight("q8", 70, 512, 19)
    _, b = weight("q8", 70, 512, 20)
    x = torch.from_numpy(make_x(M, 512, seed=21)).cuda()
    h, both = (torch.full((M, 70), float("nan"), device="cuda") for _ in range(2))
    sq.matmul_swiglu_dev(a, b, x.data_ptr(), M, 512, h.data_ptr())
    p = both.data_ptr()
    sq.matmul_swiglu_dev(a, b, x.data_ptr(), M, 512, p, p if over == "gate" else 0, p if over == "up" else 0)
    torch.cuda.synchronize()
    assert torch.isfinite(h).all() and torch.equal(both, h)


@pytest.mark.parametrize("qtype", QTYPES)
@pytest.mark.parametrize("K,M", [(768, 7), (2048, 7), (4096, 32)])
def test_as_close_to_64_bits_as_the_gemv(qtype, K, M):
    # the min joins its block's term before the scale: apart, the two would enter the sum
    # at their own size (1.8 times the GEMV's error)
    N = 512
    rng = np.random.default_rng(K)
    raw, W = _power_of_two_weight(qtype, N, K, rng)
    if qtype in ("q4_1", "q5k1"):
        # mins that centre the weights on zero, as a trained layer's do
        d = raw.reshape(-1)[:N * K // 32 * 20].reshape(N, K // 32, 20)
        s = d[..., 0:2].copy().view(np.float16)[..., 0].astype(np.float64)
        m0 = d[..., 2:4].copy().view(np.float16)[..., 0].astype(np.float64)
        m = s * (-7.5 if qtype == "q4_1" else -15.5)
        d[..., 2:4] = m.astype(np.float16).view(np.uint8).reshape(N, K // 32, 2)
        W = W + (m - m0)[..., None]
    w = sq.DeviceWeight.from_quant(sq.QuantWeight(qtype, np.ascontiguousarray(raw).reshape(-1), K // 32, N, K))
    # activations that quantize exactly (127 in every block)
    x = rng.integers(-126, 127, (M, K // 32, 32)).astype(np.float32)
    x[..., 0] = 127
    x = (x * 2.0 ** rng.integers(-6, 1, (M, K // 32, 1))).astype(np.float32).reshape(M, K)
    ref = x.astype(np.float64) @ W.reshape(N, K).T
    err = lambda y: np.linalg.norm(y - ref) / np.linalg.norm(ref)
    e = err(run(w, x))
    sq.set_param("gemm_min_rows", 1 << 20)
    g = err(run(w, x))
    assert e <= 1.05 * g, (e, g)


@pytest.mark.parametrize("qtype", ["q4", "q5k1"])
@pytest.mark.parametrize("N,M", [(2048, 32), (2049, 32), (3072, 24), (3072, 32), (3073, 24), (4096, 18), (4096, 19), (4097, 9)])
def test_splits_of_wider_weights_give_the_bits_of_one_launch(qtype, N, M):
    # alone (in K splits where the rule says so) and beside another weight (one launch)
    K = 2304
    _, a = weight(qtype, N, K, 22)
    _, b = weight(qtype, 33, K, 23)
    x = torch.from_numpy(make_x(M, K, seed=24)).cuda()
    alone, ya = (torch.full((M, N), float("nan"), device="cuda") for _ in range(2))
    yb = torch.empty((M, 33), device="cuda")
    sq.matmul_dev(a, x.data_ptr(), M, K, alone.data_ptr())
    sq.matmul_multi_dev([a, b], x.data_ptr(), M, K, [ya.data_ptr(), yb.data_ptr()])
    torch.cuda.synchronize()
    assert torch.isfinite(alone).all() and torch.equal(alone, ya)
