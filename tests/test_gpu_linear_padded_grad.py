"""bf16 Linear backward where a gradient row is no whole number of 16 bytes: the pass that pads it, sums
the bias gradient and applies the activation, the products that read the padded rows, the reduction
split over workgroups, and a product whose last round goes as its own."""
import numpy as np
import pytest
import torch

from util import assert_close, bf16_round, rng, to_dev, to_np

pytestmark = pytest.mark.gpu
BT = torch.bfloat16


def backward(ffk, oracle, batch, in_dim, out_dim, act, accumulate, shrink):
    g = rng(batch + in_dim * 3 + out_dim * 5 + accumulate)
    x, w, y, dy = (bf16_round(g.standard_normal(s)) for s in ((batch, in_dim), (out_dim, in_dim), (batch, out_dim), (batch, out_dim)))
    grad = np.where(y > 0, dy, 0.0) if act == ffk.ACT_RELU else dy
    old = [bf16_round(g.standard_normal(s)) for s in ((batch, in_dim), (out_dim, in_dim), (out_dim,))]
    dx, dw, db = (to_dev(o, torch, BT) for o in old)
    need = ffk.lib().ffk_linear_backward_workspace_bytes(ffk.BF16, act, 1, batch, out_dim)
    ws = torch.full((need + 256,), 0x7f, dtype=torch.uint8, device="cuda")  # (bytes 7f7f: a huge bf16)
    # `shrink`: a caller that brings what the operator needs without a padded gradient
    least = need - (-(-batch * ((out_dim + 63) // 64 * 64) * 2 // 256) * 256)
    if act != ffk.ACT_NONE:
        least += -(-batch * out_dim * 2 // 256) * 256
    ffk.linear_backward(to_dev(y, torch, BT), to_dev(dy, torch, BT), to_dev(x, torch, BT), to_dev(w, torch, BT), dx, dw, db,
                        activation=act, accumulate=accumulate, workspace=ws[:least if shrink else need])
    assert bool((ws[need:] == 0x7f).all())
    want = [oracle.gemm_f64(grad, w, False, False), oracle.gemm_f64(grad, x, True, False), grad.astype(np.float64).sum(0)]
    for name, got, ref, before in zip(("dx", "dw", "db"), (dx, dw, db), want, old):
        # exact products, fp32 accumulation, one bf16 rounding at the store
        assert_close(to_np(got), ref + before if accumulate else ref, 2.0 ** -8, name)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("act", ["none", "relu"])
@pytest.mark.parametrize("shape", [(1, 8, 9), (33, 136, 1001), (257, 264, 65), (130, 136, 9001), (300, 256, 263)])
def test_padded_gradient(ffk, oracle, shape, act, accumulate):
    print("padded gradient", shape, act, accumulate, flush=True)
    backward(ffk, oracle, *shape, {"none": ffk.ACT_NONE, "relu": ffk.ACT_RELU}[act], accumulate, False)


@pytest.mark.parametrize("act", ["none", "relu"])
def test_workspace_without_room_for_the_padding(ffk, oracle, act):
    backward(ffk, oracle, 65, 72, 501, {"none": ffk.ACT_NONE, "relu": ffk.ACT_RELU}[act], False, True)


@pytest.mark.parametrize("ta,tb,M,N", [(False, True, 2048, 8457), (False, True, 8457, 2048), (True, False, 8456, 2048)])
def test_whole_rounds_and_the_rest(ffk, ta, tb, M, N):
    """264 tiles of 256 x 256 on 256 CUs."""
    print("whole rounds", M, N, ta, tb, flush=True)
    K = 1024
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    a, b = (torch.randn(s, generator=gen, device="cuda").to(BT) for s in (((K, M) if ta else (M, K)), ((N, K) if tb else (K, N))))
    buf = torch.full((M * N + 16,), 7.0, dtype=BT, device="cuda")
    c = buf[8:8 + M * N].view(M, N)
    ffk.gemm(a, b, c, ta, tb)
    want = torch.matmul((a.t() if ta else a).float(), (b.t() if tb else b).float())
    err = (c.float() - want).abs()
    # one bf16 rounding, and fp32 sums of 1024 products of unit variance in another order
    assert bool((err <= 2.0 ** -8 * want.abs() + 1e-3).all()), float(err.max())
    assert bool((buf[:8] == 7.0).all()) and bool((buf[8 + M * N:] == 7.0).all())
