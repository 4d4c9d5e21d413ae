"""bf16 products on 32x32 tiles, whose four waves split the reduction: the edges of the tile, reductions that leave
waves without a part, bias and activation behind the sum of the waves."""
import pytest
import torch

from util import assert_close, to_np

pytestmark = pytest.mark.gpu
BT = torch.bfloat16


@pytest.fixture
def tile32(ffk):
    ffk.set_option(ffk.OPTION_GEMM_VARIANT, 32)
    yield
    ffk.set_option(ffk.OPTION_GEMM_VARIANT, 0)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("mnk", [(32, 32, 32), (8, 8, 8), (40, 72, 136), (31, 64, 96), (96, 40, 2056), (64, 1000, 520), (200, 264, 128)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_edges(ffk, tile32, ta, tb, mnk, accumulate):
    M, N, K = mnk
    if ta and M % 8 != 0:
        M += 8 - M % 8
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = (torch.randn(s, generator=gen, device="cuda").to(BT) for s in ((K, M) if ta else (M, K), (N, K) if tb else (K, N)))
    assert ffk.gemm_kernel_name(ffk.BF16, ta, tb, M, N, K).startswith("gemm_bf16_pipe_kernel<32,32,")
    buf = torch.randn(M * N + 16, generator=gen, device="cuda").to(BT)
    before = buf.clone()
    C = buf[8:8 + M * N].view(M, N)
    want = (A.t() if ta else A).double() @ (B.t() if tb else B).double()
    ffk.gemm(A, B, C, ta, tb, accumulate=accumulate)
    # exact products, fp32 accumulation, one bf16 rounding at the store
    assert_close(to_np(C), to_np(want + before[8:8 + M * N].view(M, N).double() if accumulate else want), 2.0 ** -8, "C")
    assert torch.equal(buf[:8], before[:8]) and torch.equal(buf[8 + M * N:], before[8 + M * N:])


@pytest.mark.parametrize("act", ["NONE", "RELU", "GELU"])
@pytest.mark.parametrize("shape", [(33, 72, 45), (64, 256, 96), (7, 1032, 200)])
def test_bias_and_activation(ffk, tile32, act, shape):
    B, I, O = shape
    gen = torch.Generator(device="cuda").manual_seed(B)
    x, w, b = (torch.randn(s, generator=gen, device="cuda").to(BT) for s in ((B, I), (O, I), (O,)))
    w *= 0.125  # exact
    want = x.double() @ w.double().t() + b.double()
    want = {"NONE": want, "RELU": want.clamp(min=0), "GELU": torch.nn.functional.gelu(want)}[act]
    y = ffk.linear_forward(x, w, b, activation=getattr(ffk, "ACT_" + act))
    assert_close(to_np(y), to_np(want), 2.0 ** -8, "y")


def test_values_next_to_the_edge_stay_out(ffk, tile32):
    M, N, K = 72, 136, 72
    A, B = torch.ones((M, K), device="cuda", dtype=BT), torch.ones((N, K), device="cuda", dtype=BT)
    A[5, 0] = float("inf")  # follows row 4's last element in memory
    C = torch.empty((M, N), device="cuda", dtype=BT)
    ffk.gemm(A, B, C, False, True)
    rows = torch.isinf(C).any(1)
    assert bool(rows[5]) and int(rows.sum()) == 1 and not bool(torch.isnan(C).any())
