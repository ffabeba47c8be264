"""Calls whose workspace cannot be had (here: is limited) take the kernels that need
less of it, as long as there are some."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import sllm_qmm as sq

from _helpers import make_raw, make_x
from test_gpu_attention import Model
from test_gpu_attention_prompt import _run
from test_gpu_kquant_native import make_kq

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _params():
    yield
    for p in ("workspace_max_mb", "gemm_min_rows"):
        sq.set_param(p, 0)


def _matmul(w, x):
    xd = torch.from_numpy(x).cuda()
    y = torch.full((x.shape[0], w.rows), float("nan"), device="cuda")
    sq.matmul_dev(w, xd.data_ptr(), *x.shape, y.data_ptr())
    return y


def test_prompt_attention_falls_back_to_the_split_kernel():
    # q rows of 4.7 MiB, the matrix cores' states of several times that
    rng = np.random.default_rng(1)
    m = Model(32, 8, 128, 0, rng)
    seq = 300
    q, k, v = (rng.normal(size=(seq, n * 128)).astype(np.float32) for n in (32, 8, 8))
    ck, cv = (np.zeros((8, seq, 128), np.float32) for _ in range(2))
    full = _run(m, q, k, v, ck, cv, seq, 0)
    split = _run(m, q, k, v, ck, cv, seq, 0, offset=1)  # an output off 16 bytes
    sq.set_param("workspace_max_mb", 8)
    limited = _run(m, q, k, v, ck, cv, seq, 0)
    assert np.array_equal(limited.view(np.uint32), split.view(np.uint32))
    assert not np.array_equal(limited, full)
    sq.set_param("workspace_max_mb", 2)
    with pytest.raises(sq.SllmError) as e:
        _run(m, q, k, v, ck, cv, seq, 0)
    assert e.value.status == 5


def test_kquant_prompts_fall_back_to_the_gemv_and_int8_ones_fail():
    K, M = 4096, 256  # the split activations alone: 6 MiB
    w = sq.load_weight_f32_direct(11, make_kq(11, 64, K, 2), 64, K)
    x = make_x(M, K, seed=3)
    full = _matmul(w, x)
    sq.set_param("gemm_min_rows", 1 << 20)
    gemv = _matmul(w, x)
    sq.set_param("gemm_min_rows", 0)
    sq.set_param("workspace_max_mb", 5)
    assert torch.equal(_matmul(w, x), gemv) and not torch.equal(gemv, full)
    w8 = sq.DeviceWeight.from_quant(sq.QuantWeight("q8", make_raw("q8", 64, K, seed=4), K // 32, 64, K))
    sq.set_param("workspace_max_mb", 1)
    with pytest.raises(sq.SllmError) as e:
        _matmul(w8, x)
    assert e.value.status == 5
    sq.set_param("workspace_max_mb", 0)
    assert torch.isfinite(_matmul(w8, x)).all()
