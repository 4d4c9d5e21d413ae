"""LayerNorm, Softmax and Dropout on rows that are neither whole 16-byte vectors nor aligned: the
register-resident kernels with any-address accesses, at the edges of their row configurations."""
import numpy as np
import pytest
import torch

from util import BF16_RTOL, assert_close, bf16_round, rng, to_dev, to_np

pytestmark = pytest.mark.gpu
# lengths around one vector, one wave's row, one workgroup's row, several vectors a lane
LENGTHS = [1, 3, 9, 257, 511, 1001, 1027, 2051, 4099, 8191]


def inputs(dtype, M, N, scale=1.0):
    g = rng(M * 31 + N)
    rnd = bf16_round if dtype == "bf16" else (lambda a: np.asarray(a, np.float32))
    td = torch.bfloat16 if dtype == "bf16" else torch.float32
    return g, rnd, td, 2e-5 if dtype == "fp32" else BF16_RTOL


def guarded(t):
    """t's values between guard elements, its first element off 16-byte alignment."""
    buf = torch.full((t.numel() + 16,), 7.0, dtype=t.dtype, device=t.device)
    v = buf[7:7 + t.numel()].view(t.shape)
    v.copy_(t)
    return buf, v


def intact(buf):
    return bool((buf[:7] == 7.0).all()) and bool((buf[-9:] == 7.0).all())


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("N", LENGTHS)
def test_layer_norm_any_length(ffk, oracle, dtype, N):
    M = 1 if N == 3 else 2053 if N == 9 else 13
    print("layer_norm any length", (M, N), dtype, flush=True)
    g, rnd, td, rtol = inputs(dtype, M, N)
    x, dy, dx0 = rnd(g.standard_normal((M, N)) + 0.3), rnd(g.standard_normal((M, N))), rnd(g.standard_normal((M, N)))
    gamma, beta = rnd(1 + 0.1 * g.standard_normal((N,))), rnd(0.1 * g.standard_normal((N,)))
    y_ref, mean_ref, rstd_ref = oracle.layer_norm_forward(x, gamma, beta, 1e-2)
    xd, dyd, gd, bd = (to_dev(a, torch, td) for a in (x, dy, gamma, beta))
    ybuf, y = guarded(torch.zeros_like(xd))
    _, mean, rstd = ffk.layer_norm_forward(xd, gd, bd, 1e-2, out=y)
    assert intact(ybuf)
    assert_close(to_np(y), y_ref, rtol, "y")
    assert_close(to_np(mean), mean_ref, 2e-5, "mean")
    assert_close(to_np(rstd), rstd_ref, 2e-5, "rstd")
    want, dg_ref, db_ref = oracle.layer_norm_backward(dy, x, mean_ref, rstd_ref, gamma, dx_init=dx0)
    dxbuf, dx = guarded(to_dev(dx0, torch, td))
    dg, db = torch.zeros((N,), dtype=td, device="cuda"), torch.zeros((N,), dtype=td, device="cuda")
    ffk.layer_norm_backward(dyd, xd, mean, rstd, gd, dx, dg, db, accumulate=ffk.LN_ACC_INPUT)
    assert intact(dxbuf)
    assert_close(to_np(dx), want, rtol * 2, "dx accumulate")
    assert_close(to_np(dg), dg_ref, rtol * 2, "dgamma")
    assert_close(to_np(db), db_ref, rtol * 2, "dbeta")
    # without a workspace: the kernels that need none
    dg2, db2 = torch.zeros_like(dg), torch.zeros_like(db)
    if N % (4 if dtype == "fp32" else 8) != 0:
        ffk.check(ffk.lib().ffk_layer_norm_backward(ffk.current_stream(), ffk.dtype_of(xd), dyd.data_ptr(), xd.data_ptr(),
                                                    mean.data_ptr(), rstd.data_ptr(), gd.data_ptr(), None, dg2.data_ptr(),
                                                    db2.data_ptr(), M, N, None, 0, 0))
        assert_close(to_np(dg2), dg_ref, rtol * 2, "dgamma without workspace")
        assert_close(to_np(db2), db_ref, rtol * 2, "dbeta without workspace")


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("N", LENGTHS)
def test_softmax_any_length(ffk, oracle, dtype, N):
    M = 11
    print("softmax any length", (M, N), dtype, flush=True)
    g, rnd, td, rtol = inputs(dtype, M, N)
    x, dy = rnd(4 * g.standard_normal((M, N))), rnd(g.standard_normal((M, N)))
    ybuf, y = guarded(torch.zeros((M, N), dtype=td, device="cuda"))
    ffk.softmax_forward(to_dev(x, torch, td), M, N, 1, out=y)
    assert intact(ybuf)
    assert_close(to_np(y), oracle.softmax_forward(x, M, N, 1), rtol, "y")
    dxbuf, dx = guarded(torch.zeros((M, N), dtype=td, device="cuda"))
    ffk.softmax_backward(y, to_dev(dy, torch, td), M, N, 1, dx=dx)
    assert intact(dxbuf)
    assert_close(to_np(dx), oracle.softmax_backward(to_np(y), dy, M, N, 1), rtol, "dx")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 5, 7, 8, 2049, 2047 * 8 + 3])
@pytest.mark.parametrize("accumulate", [False, True])
def test_dropout_tail(ffk, oracle, dtype, n, accumulate):
    """The elements behind the last whole vector, in the same launch."""
    print("dropout tail", n, dtype, flush=True)
    g = rng(n)
    x, y0 = (bf16_round(g.standard_normal(n)) for _ in range(2))
    xd = to_dev(x, torch, dtype)
    buf = torch.full((n + 8,), 7.0, dtype=dtype, device="cuda")
    y = buf[:n]
    y.copy_(to_dev(y0, torch, dtype))
    ffk.dropout_backward(xd, 0.25, 77, 16, dx=y, accumulate=accumulate)
    want = ffk.dropout_forward(xd, 0.25, 77, 16)
    mask = oracle.dropout_mask(n, 0.25, 77, 16)
    assert bool(((want != 0).cpu().numpy() == (mask.astype(bool) & (x != 0))).all())
    expect = (want.float() + (to_dev(y0, torch, dtype).float() if accumulate else 0)).to(dtype)
    assert_close(to_np(y), to_np(expect), 2.0 ** -8, "dx")
    assert bool((buf[n:] == 7.0).all())
