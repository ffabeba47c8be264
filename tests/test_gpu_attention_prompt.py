"""GPU tests of the prompt attention on the matrix cores (several query rows):
edges of its 32-row blocks, 32-position tiles, chunks and head sizes, against
the oracle within the bound of test_gpu_attention.py (the float32 summation
error of scores and sums; their association does not enter it)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import sllm_qmm as sq

from test_gpu_attention import Model, dev_view, run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KV,dk,half,seq,cache_len", [
    (4, 1, 128, 64, 8, 0), (4, 1, 128, 64, 33, 31), (6, 2, 64, 32, 64, 0), (6, 2, 64, 32, 65, 95),
    (5, 5, 32, 16, 40, 1), (8, 1, 96, 48, 31, 64), (3, 3, 80, 40, 97, 0), (2, 2, 100, 20, 32, 33),
    (7, 1, 4, 2, 9, 30), (8, 2, 128, 64, 10, 700), (2, 1, 124, 62, 200, 0)])
def test_shapes(H, KV, dk, half, seq, cache_len):
    rng = np.random.default_rng(H * 100 + dk + seq)
    run_case(Model(H, KV, dk, half, rng), seq, cache_len, rng)


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
    m = Model(4, 2, 64, 32, rng)
    seq, cl = 80, 20
    q, k, v = (rng.normal(size=(seq, n * 64)).astype(np.float32) for n in (4, 2, 2))
    ck, cv = (rng.normal(size=(2, cl + seq, 64)).astype(np.float32) for _ in range(2))
    a = _run(m, q, k, v, ck, cv, seq, cl)
    bad = v.copy()
    bad[37, 5] = np.inf          # kv head 0, dimension 5
    bad[50, 64 + 63] = np.nan    # kv head 1, dimension 63
    bad[51, 64 + 2] = -np.inf
    b = _run(m, q, k, bad, ck, cv, seq, cl)
    hit = np.zeros_like(a, bool)
    hit[37:, :2, 5] = hit[50:, 2:, 63] = hit[51:, 2:, 2] = True
    assert np.array_equal(a[~hit].view(np.uint32), b[~hit].view(np.uint32))
    assert not np.isfinite(b[hit]).any()
    assert (b[37:, :2, 5] == np.inf).all() and (b[51:, 2:, 2] == -np.inf).all()


def test_an_output_off_16_bytes_is_taken_as_before():
    rng = np.random.default_rng(4)
    m = Model(4, 2, 64, 32, rng)
    seq, cl = 40, 9
    q, k, v = (rng.normal(size=(seq, n * 64)).astype(np.float32) for n in (4, 2, 2))
    ck, cv = (rng.normal(size=(2, cl + seq, 64)).astype(np.float32) for _ in range(2))
    a = _run(m, q, k, v, ck, cv, seq, cl)
    b = _run(m, q, k, v, ck, cv, seq, cl, offset=1)
    assert np.abs(a - b).max() <= 1e-5 * np.abs(a).max()  # two associations of the same float32 sums


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
