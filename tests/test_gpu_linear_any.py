"""bf16 Linear and products over rows of any length at any address: the register-staged tiles at their edges,
and the backward as jobs of one launch, with whole and with split reductions."""
import numpy as np
import pytest
import torch

from util import assert_close, to_np

pytestmark = pytest.mark.gpu
BT = torch.bfloat16
NONE, RELU, SIGMOID, TANH = "NONE", "RELU", "SIGMOID", "TANH"


def somewhere(gen, *shape, shift=1):
    """A random tensor that begins `shift` elements past a 16-byte boundary, between NaNs."""
    n = int(np.prod(shape))
    buf = torch.full((n + 64,), float("nan"), dtype=BT, device="cuda")
    t = buf[16 + shift:16 + shift + n].view(shape)
    t.copy_(torch.randn(shape, generator=gen, device="cuda"))
    return buf, t


def intact(buf, t, shift=1):
    n = t.numel()
    return bool(buf[:16 + shift].isnan().all()) and bool(buf[16 + shift + n:].isnan().all())


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("mnk", [(300, 129, 65), (65, 200, 259), (513, 3, 2001), (7, 4001, 130), (5, 5000, 100), (1300, 1500, 63),
                                 (2100, 2051, 71), (2049, 2047, 191)])
def test_products(ffk, ta, tb, mnk):
    """One short of, at and one past the 64 and 128 wide tiles and the 64 deep k-tiles, and rows of fewer than 16 bytes."""
    M, N, K = mnk
    print("gemm any", mnk, ta, tb, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    (_, A), (_, B) = somewhere(gen, *((K, M) if ta else (M, K))), somewhere(gen, *((N, K) if tb else (K, N)))
    cb, C = somewhere(gen, M, N)
    ffk.gemm(A, B, C, ta, tb)
    want = (A.t() if ta else A).double() @ (B.t() if tb else B).double()
    # one rounding to bf16 of an fp32 sum: half a unit in the last of 8 bits
    assert_close(to_np(C), to_np(want), 2.0 ** -8, "C")
    assert intact(cb, C)


# batch, in, out: one tile and its edges, rows of fewer than 16 bytes, both reductions split, each alone, and the large tiles
SHAPES = [(1, 1, 1), (3, 5, 7), (33, 72, 40), (64, 64, 64), (65, 63, 129), (127, 65, 1), (17, 212, 4185), (2972, 89, 65),
          (1100, 200, 1301), (640, 2263, 1700)]


@pytest.mark.parametrize("act", [NONE, RELU, SIGMOID, TANH])
@pytest.mark.parametrize("shape", SHAPES)
def test_linear(ffk, act, shape):
    B, I, O = shape
    print("linear any", shape, act, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B + I * 3 + O * 5)
    code = getattr(ffk, "ACT_" + act)
    (_, x), (_, w), (_, y), (_, dy) = (somewhere(gen, *s) for s in ((B, I), (O, I), (B, O), (B, O)))
    yd, g = y.double(), dy.double()
    g = {NONE: g, RELU: torch.where(yd > 0, g, 0.0), SIGMOID: g * yd * (1 - yd), TANH: g * (1 - yd * yd)}[act].to(BT).double()
    want = {"dx": g @ w.double(), "dw": g.t() @ x.double(), "db": g.sum(0)}
    outs = {"dx": somewhere(gen, B, I), "dw": somewhere(gen, O, I), "db": somewhere(gen, O)}
    for accumulate in (0, 7):
        before = {k: t.double() for k, (_, t) in outs.items()}
        ffk.linear_backward(y, dy, x, w, *(outs[k][1] for k in ("dx", "dw", "db")), activation=code, accumulate=accumulate)
        for k, (buf, t) in outs.items():
            # g is rounded to bf16 from fp32, where the reference's double may round the other way: a unit of a
            # few terms beside one rounding of the sum
            tol = 2.0 ** -8 if act in (NONE, RELU) else 2.0 ** -7
            assert_close(to_np(t), to_np(want[k] + before[k] if accumulate else want[k]), tol, "%s %s" % (k, accumulate))
            assert intact(buf, t), k
    # each gradient alone: the same bits
    for keep in (("dx",), ("dw",), ("dx", "db")):
        again = {k: torch.empty_like(outs[k][1]) if k in keep else None for k in outs}
        full = {k: torch.empty_like(t) for k, (_, t) in outs.items()}
        ffk.linear_backward(y, dy, x, w, *(again[k] for k in ("dx", "dw", "db")), activation=code, accumulate=0)
        ffk.linear_backward(y, dy, x, w, *(full[k] for k in ("dx", "dw", "db")), activation=code, accumulate=0)
        assert all(torch.equal(again[k], full[k]) for k in keep), keep


def test_gradient_written_over_the_output_gradient(ffk):
    """A caller may let the input gradient take the output gradient's memory behind an activation."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, w, y, dy = (torch.randn(s, generator=gen, device="cuda").to(BT) for s in ((100, 72), (72, 72), (100, 72), (100, 72)))
    apart = [torch.empty_like(x), torch.empty_like(w), torch.empty(72, dtype=BT, device="cuda")]
    ffk.linear_backward(y, dy, x, w, *apart, activation=ffk.ACT_RELU, accumulate=0)
    over = dy.clone()
    got = [over, torch.empty_like(w), torch.empty(72, dtype=BT, device="cuda")]
    ffk.linear_backward(y, over, x, w, *got, activation=ffk.ACT_RELU, accumulate=0)
    for a, b, name in zip(apart, got, ("dx", "dw", "db")):
        assert_close(to_np(b), to_np(a), 2.0 ** -7, name)


@pytest.mark.parametrize("shape", [(64, 128, 40), (96, 128, 256), (65, 63, 129)])
def test_the_layer_option_leaves_a_linear_alone(ffk, shape):
    """What makes an encoder layer run one kernel per operator is no switch of the operators: the same bits either way."""
    B, I, O = shape
    gen = torch.Generator(device="cuda").manual_seed(B)
    x, w, dy = (torch.randn(s, generator=gen, device="cuda").to(BT) for s in ((B, I), (O, I), (B, O)))
    got = []
    for value in (0, 1):
        out = [torch.empty_like(x), torch.empty_like(w), torch.empty(O, dtype=BT, device="cuda")]
        ffk.set_option(ffk.OPTION_LAYER_UNFUSED, value)
        try:
            ffk.linear_backward(None, dy, x, w, *out, accumulate=0)
        finally:
            ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 0)
        got.append(out)
    assert all(torch.equal(a, b) for a, b in zip(*got))
