"""bf16 products on 256x128 tiles: the edges of the tile, whole tiles, ragged reductions, and the same bits as on the
128x128 tiles that they take the place of, also with the operators of an encoder layer on their store."""
import numpy as np
import pytest
import torch

from layer_oracle import make_params
from test_gpu_encoder_layer import run_device
from util import assert_close, bf16_round, rng, to_np

pytestmark = pytest.mark.gpu
BT = torch.bfloat16


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("mnk", [(2304, 2048, 64), (1379, 3072, 200), (264, 12008, 72), (16504, 136, 8), (2056, 2056, 1032)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_edges(ffk, ta, tb, mnk, accumulate):
    M, N, K = mnk
    if ta and M % 8 != 0:
        M += 8 - M % 8
    print(M, N, K, ta, tb, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = (torch.randn(s, generator=gen, device="cuda").to(BT) for s in ((K, M) if ta else (M, K), (N, K) if tb else (K, N)))
    assert ffk.gemm_kernel_name(ffk.BF16, ta, tb, M, N, K).startswith("gemm_bf16_pipe_kernel<256,128,")
    buf = torch.randn(M * N + 16, generator=gen, device="cuda").to(BT)
    before = buf.clone()
    C = buf[8:8 + M * N].view(M, N)
    want = (A.t() if ta else A).double() @ (B.t() if tb else B).double()
    ffk.gemm(A, B, C, ta, tb, accumulate=accumulate)
    # exact products, fp32 accumulation, one bf16 rounding at the store
    assert_close(to_np(C), to_np(want + before[8:8 + M * N].view(M, N).double() if accumulate else want), 2.0 ** -8, "C")
    assert torch.equal(buf[:8], before[:8]) and torch.equal(buf[8 + M * N:], before[8 + M * N:])
    other = before.clone()
    ffk.set_option(ffk.OPTION_GEMM_VARIANT, 128)
    try:
        ffk.gemm(A, B, other[8:8 + M * N].view(M, N), ta, tb, accumulate=accumulate)
    finally:
        ffk.set_option(ffk.OPTION_GEMM_VARIANT, 0)
    assert torch.equal(buf, other)


def test_odd_width_with_bias_and_activation(ffk):
    B, I, O = 2050, 72, 2051
    gen = torch.Generator(device="cuda").manual_seed(B)
    x, w, b = (torch.randn(s, generator=gen, device="cuda").to(BT) for s in ((B, I), (O, I), (O,)))
    w *= 0.125  # exact
    y = ffk.linear_forward(x, w, b, activation=ffk.ACT_RELU)
    assert_close(to_np(y), to_np((x.double() @ w.double().t() + b.double()).clamp(min=0)), 2.0 ** -8, "y")


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("batch,seq", [(5, 260), (8, 160)])
def test_operators_on_the_store(ffk, gelu, batch, seq):
    d_ff = 3072 if batch == 5 else 3328  # 264 tiles of 128 x 128 with ragged rows, 260 of whole ones
    cfg = dict(batch=batch, seq=seq, d_model=128, heads=2, d_ff=d_ff, p=0.1, seed=3, eps=1e-5, scale=0.125, causal=False,
               pre_ln=True, gelu=gelu)
    print(cfg, flush=True)
    g = rng(seq)
    params = make_params(g, cfg, bf16_round)
    x, dy = (bf16_round(g.standard_normal((batch, seq, 128))) for _ in range(2))
    y, dx, grads = run_device(ffk, cfg, params, x, dy)
    ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 1)
    try:
        y1, dx1, _ = run_device(ffk, cfg, params, x, dy)
    finally:
        ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 0)
    # the same operands, operators and order of sums, in one kernel or two
    assert np.array_equal(y, y1) and np.array_equal(dx, dx1)
    assert np.abs(grads["b1"]).max() > 0
