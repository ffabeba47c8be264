"""GPU tests of the prompt attention on the matrix cores (several query rows):
edges of its 32-row blocks, 32-position tiles, chunks and head sizes, against
the oracle within the bound of test_gpu_attention.py (the float32 summation
error of scores and sums; their association does not enter it). The shapes lie
above the line from which a prompt takes that kernel (test_the_line_between_the_kernels):
512 pairs of row and kv head, up to 1536 where two tiles of 64 hold the positions."""
from __future__ import annotations

import gc

import numpy as np
import pytest
import torch

import sllm_qmm as sq

from test_gpu_attention import Model, dev_view, run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,dk,half,seq,cache_len,norms", [
    (4, 1, 128, 64, 520, 0, False), (4, 1, 128, 64, 545, 31, False), (32, 32, 64, 32, 65, 31, False),
    (6, 2, 64, 32, 320, 95, True), (8, 8, 32, 16, 97, 1, False), (6, 3, 20, 10, 300, 0, False), (8, 8, 96, 48, 129, 64, False),
    (3, 3, 80, 40, 260, 0, True), (7, 1, 100, 20, 520, 33, False), (6, 2, 36, 18, 400, 31, False), (8, 2, 128, 64, 300, 700, True),
    (14, 2, 124, 62, 290, 5, False), (16, 4, 128, 32, 170, 0, True), (24, 24, 48, 24, 64, 2, False), (2, 2, 4, 2, 1030, 0, False)])
def test_shapes(H, KV, dk, half, seq, cache_len, norms):
    rng = np.random.default_rng(H * 100 + dk + seq)
    run_case(Model(H, KV, dk, half, rng, bias=norms, qk=norms), seq, cache_len, rng)


def _run(m, q, k, v, ck, cv, seq, cache_len, offset=0):
    kv = sq.KVCache(1, m.KV, m.dk, cache_len + seq)
    for ptr, src in zip(kv.data(0), (ck, cv)):
        dev_view(ptr, src.size).copy_(torch.from_numpy(src.reshape(-1)))
    kv.set_length(cache_len)
    out = torch.full((seq * m.H * m.dk + 4,), float("nan"), device="cuda")[offset:offset + seq * m.H * m.dk]
    d = [torch.from_numpy(a).cuda() for a in (q, k, v)]
    sq.attention_dev(kv, 0, m.params, *[t.data_ptr() for t in d], seq, cache_len, out.data_ptr())
    torch.cuda.synchronize()
    return out.cpu().numpy().reshape(seq, m.H, m.dk)


def test_a_later_rows_infinite_value_does_not_reach_earlier_rows():
    # non-finite v elements of position p: rows before p equal the run without
    # them bit for bit; from p on exactly the elements' dimensions are non-finite
    rng = np.random.default_rng(3)
    m = Model(16, 8, 64, 32, rng)
    seq, cl = 170, 20
    q, k, v = (rng.normal(size=(seq, n * 64)).astype(np.float32) for n in (16, 8, 8))
    ck, cv = (rng.normal(size=(8, cl + seq, 64)).astype(np.float32) for _ in range(2))
    a = _run(m, q, k, v, ck, cv, seq, cl)
    bad = v.copy()
    bad[37, 5] = np.inf          # kv head 0, dimension 5
    bad[50, 64 + 63] = np.nan    # kv head 1, dimension 63
    bad[51, 64 + 2] = -np.inf
    b = _run(m, q, k, bad, ck, cv, seq, cl)
    hit = np.zeros_like(a, bool)
    hit[37:, :2, 5] = hit[50:, 2:4, 63] = hit[51:, 2:4, 2] = True
    assert np.array_equal(a[~hit].view(np.uint32), b[~hit].view(np.uint32))
    assert not np.isfinite(b[hit]).any()
    assert (b[37:, :2, 5] == np.inf).all() and (b[51:, 2:4, 2] == -np.inf).all()


@pytest.mark.parametrize("H,KV,dk,seq,cl", [(16, 8, 64, 200, 9), (64, 64, 8, 1030, 0)])
def test_an_output_off_16_bytes_takes_the_split_kernel(H, KV, dk, seq, cl):
    # (1030 rows of 64 kv heads: more than the 65535 of its grid, so in two launches)
    rng = np.random.default_rng(4)
    m = Model(H, KV, dk, dk // 2, rng)
    q, k, v = (rng.normal(size=(seq, n * dk)).astype(np.float32) for n in (H, KV, KV))
    ck, cv = (rng.normal(size=(KV, cl + seq, dk)).astype(np.float32) for _ in range(2))
    a = _run(m, q, k, v, ck, cv, seq, cl)
    b = _run(m, q, k, v, ck, cv, seq, cl, offset=1)
    assert not np.array_equal(a, b)
    assert np.abs(a - b).max() <= 1e-5 * np.abs(a).max()  # two associations of the same float32 sums


def test_capture_without_workspace_takes_the_split_kernel():
    rng = np.random.default_rng(5)
    m = Model(32, 8, 128, 64, rng)
    seq = 300
    q, k, v = (rng.normal(size=(seq, n * 128)).astype(np.float32) for n in (32, 8, 8))
    z = np.zeros((8, seq, 128), np.float32)
    split = _run(m, q, k, v, z, z, seq, 0, offset=1)
    kv = sq.KVCache(1, 8, 128, seq)
    d = [torch.from_numpy(t).cuda() for t in (q, k, v)]
    out = torch.empty((seq, 32, 128), device="cuda")
    # a workspace of 8 MiB holds the q rows (4.7), not the chunks' states
    s = torch.cuda.Stream()
    sq.set_param("workspace_max_mb", 8)
    sq.workspace_reserve(s.cuda_stream, 8 << 20)
    g = torch.cuda.CUDAGraph()
    gc.collect()
    with torch.cuda.graph(g, stream=s):
        sq.attention_dev(kv, 0, m.params, *[t.data_ptr() for t in d], seq, 0, out.data_ptr(), s.cuda_stream)
    sq.set_param("workspace_max_mb", 0)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().view(np.uint32), split.view(np.uint32))
    del g
    kv.close()


def test_weights_are_the_rounded_64_bit_exponential():
    # two cached positions, scores 0 and x <= -18 with values 0 and 1 (the rows' own
    # positions weigh 0): the sum of weights is 1 in float32, so the output is the
    # weight itself, float32(exp(float64(x)))
    rng = np.random.default_rng(8)
    m = Model(8, 8, 4, 0, rng)
    seq, cl = 600, 2
    x = np.float32(-18) - rng.uniform(0, 86, size=(seq, 8)).astype(np.float32)
    q = np.zeros((seq, 8, 4), np.float32)
    q[..., 0], q[..., 1] = 2 * x, 1  # scale 1 / sqrt(4)
    k = np.zeros((seq, 8, 4), np.float32)
    k[..., 1] = -1e6
    ck = np.zeros((8, cl + seq, 4), np.float32)
    ck[:, 1, 0] = 1
    cv = np.zeros_like(ck)
    cv[:, 1] = 1
    out = _run(m, q, k, np.ones_like(k), ck, cv, seq, cl)
    want = np.exp(x.astype(np.float64)).astype(np.float32)
    assert np.array_equal(out.view(np.uint32), np.repeat(want, 4, -1).reshape(out.shape).view(np.uint32))


def test_a_whole_tile_of_infinitely_low_scores():
    # positions 0 .. 31 overflow to -inf and weigh 0, the others weigh the same
    rng = np.random.default_rng(9)
    m = Model(8, 8, 4, 0, rng)
    seq, cl = 600, 40
    q = np.full((seq, 8, 4), 1e20, np.float32)
    ck = np.zeros((8, cl + seq, 4), np.float32)
    ck[:, :32] = -1e20
    cv = rng.normal(size=(8, cl + seq, 4)).astype(np.float32)
    v = rng.normal(size=(seq, 8, 4)).astype(np.float32)
    out = _run(m, q, np.zeros((seq, 8, 4), np.float32), v, ck, cv, seq, cl)
    seen = np.concatenate([cv[:, 32:cl].transpose(1, 0, 2), v]).astype(np.float64)
    n = 8 + np.arange(1, seq + 1)
    want = np.cumsum(seen, 0)[8:] / n[:, None, None]
    # float32 sums of up to 608 terms
    bound = (2 * 608 + 8) * 2.0 ** -24 * np.cumsum(np.abs(seen), 0)[8:] / n[:, None, None]
    assert np.all(np.abs(out - want) <= bound)


@pytest.mark.parametrize("H,KV,dk,seq,cl,flash", [
    (32, 32, 64, 48, 0, False), (32, 32, 64, 49, 0, True), (40, 40, 128, 13, 30, False), (16, 16, 80, 48, 0, False),
    (16, 16, 80, 49, 0, True), (32, 8, 128, 96, 0, False), (32, 8, 128, 97, 0, True), (32, 8, 128, 64, 65, False),
    (32, 8, 128, 65, 64, True), (64, 8, 128, 64, 0, False), (64, 8, 128, 65, 0, True), (9, 3, 64, 170, 0, False),
    (9, 3, 64, 171, 0, True), (5, 1, 256, 600, 0, False)])
def test_the_line_between_the_kernels(H, KV, dk, seq, cl, flash):
    # an output off 16 bytes always takes the split kernel: below the line both
    # outputs have its bits, above it those of two associations
    rng = np.random.default_rng(seq)
    m = Model(H, KV, dk, 0, rng)
    q, k, v = (rng.normal(size=(seq, n * dk)).astype(np.float32) for n in (H, KV, KV))
    ck, cv = (rng.normal(size=(KV, cl + seq, dk)).astype(np.float32) for _ in range(2))
    a = _run(m, q, k, v, ck, cv, seq, cl)
    b = _run(m, q, k, v, ck, cv, seq, cl, offset=1)
    assert np.abs(a - b).max() <= 1e-5 * np.abs(a).max()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)) is not flash
