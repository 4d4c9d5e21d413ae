"""Softmax rows of 321 to 512 vectors, which a workgroup takes where a wave would need eight vectors a lane: both sides of
each bound, rows of whole vectors and rows at any address."""
import numpy as np
import pytest
import torch

from util import BF16_RTOL, assert_close, bf16_round, rng, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("vectors,extra", [(320, 0), (321, 0), (321, -1), (480, 0), (481, 0), (511, 1), (512, 0), (513, 0)])
@pytest.mark.parametrize("M", [1, 7])
def test_rows_of_a_workgroup(ffk, oracle, dtype, vectors, extra, M):
    N = vectors * (4 if dtype == "fp32" else 8) + extra
    print("softmax workgroup rows", (M, N), dtype, flush=True)
    g = rng(M * 31 + N)
    rnd = bf16_round if dtype == "bf16" else (lambda a: np.asarray(a, np.float32))
    td, rtol = (torch.bfloat16, BF16_RTOL) if dtype == "bf16" else (torch.float32, 2e-5)
    x, dy = rnd(4.0 * g.standard_normal((M, N), dtype=np.float32)), rnd(g.standard_normal((M, N), dtype=np.float32))
    x[0, ::3] = -np.inf
    x64 = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    want = x64 / x64.sum(1, keepdims=True)
    y = ffk.softmax_forward(to_dev(x, torch, td), M, N, 1)
    assert_close(to_np(y), want, rtol, "y")
    yr, dy64 = to_np(y).astype(np.float64), dy.astype(np.float64)
    dx = ffk.softmax_backward(y, to_dev(dy, torch, td), M, N, 1)
    assert_close(to_np(dx), yr * (dy64 - (yr * dy64).sum(1, keepdims=True)), rtol, "dx")
