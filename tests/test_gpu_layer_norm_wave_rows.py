"""LayerNorm rows of 129 to 256 vectors: three or four vectors a lane of one wave, four waves beyond, and the row count
from which the backward takes a wave a row."""
import numpy as np
import pytest
import torch

from util import BF16_RTOL, assert_close, bf16_round, rng, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("vectors,extra", [(128, 1), (129, 0), (192, -1), (192, 0), (192, 1), (256, -1), (256, 0)])
@pytest.mark.parametrize("M", [5, 5999, 6001])
def test_rows_of_a_wave(ffk, oracle, dtype, vectors, extra, M):
    N = vectors * (4 if dtype == "fp32" else 8) + extra
    print("layer_norm wave rows", (M, N), dtype, flush=True)
    g = rng(M * 31 + N)
    rnd = bf16_round if dtype == "bf16" else (lambda a: np.asarray(a, np.float32))
    td, rtol = (torch.bfloat16, BF16_RTOL) if dtype == "bf16" else (torch.float32, 2e-5)
    x, dy, gamma, beta = (rnd(g.standard_normal(s, dtype=np.float32) * k + c)
                          for s, k, c in (((M, N), 1, 0.3), ((M, N), 1, 0), ((N,), 0.1, 1), ((N,), 0.1, 0)))
    y_ref, mean_ref, rstd_ref = oracle.layer_norm_forward(x, gamma, beta, 1e-2)
    xd, dyd, gd, bd = (to_dev(a, torch, td) for a in (x, dy, gamma, beta))
    y, mean, rstd = ffk.layer_norm_forward(xd, gd, bd, 1e-2)
    assert_close(to_np(y), y_ref, rtol, "y")
    assert_close(to_np(mean), mean_ref, 2e-5, "mean")
    assert_close(to_np(rstd), rstd_ref, 2e-5, "rstd")
    want, dg_ref, db_ref = oracle.layer_norm_backward(dy, x, mean_ref, rstd_ref, gamma)
    dx, dg, db = torch.full_like(xd, 7.0), torch.zeros_like(gd), torch.zeros_like(gd)
    ffk.layer_norm_backward(dyd, xd, mean, rstd, gd, dx, dg, db)
    assert_close(to_np(dx), want, rtol * 2, "dx")
    # M terms of unit variance: sums of about sqrt(M), whose parts of at most 12 rows a lane and then 512 workgroups are
    # added up in fp32 at an error of sqrt(524) * 2^-24 of what they hold
    assert_close(to_np(dg), dg_ref, rtol * 2, "dgamma")
    assert_close(to_np(db), db_ref, rtol * 2, "dbeta")
