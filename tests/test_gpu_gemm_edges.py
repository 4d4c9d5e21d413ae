"""bf16 GEMM at sizes that do not divide into tiles: every pipelined tile with ragged M, N and K, and
the register-staged kernel on operands whose rows start at any address."""
import numpy as np
import pytest
import torch

from util import assert_close, bf16_round, rng, to_dev, to_np

pytestmark = pytest.mark.gpu
BT = torch.bfloat16

# M, N, K: one element short of and past a tile, one row, one column group, reductions of less than
# one k-tile, of a whole one, and of a few with a remainder
ALIGNED = [(8, 8, 8), (136, 264, 72), (256, 128, 64), (248, 120, 200), (512, 520, 328), (40, 1032, 136),
           (264, 256, 1416)]
ANY = [(1, 2111, 1000), (129, 257, 65), (255, 127, 191), (131, 509, 261), (513, 33, 127)]
KINDS = [(False, True), (False, False), (True, False), (True, True)]


def product(ffk, oracle, mnk, ta, tb, accumulate):
    M, N, K = mnk
    g = rng(M * 7 + N * 3 + K)
    A = bf16_round(g.standard_normal((K, M) if ta else (M, K)))
    B = bf16_round(g.standard_normal((N, K) if tb else (K, N)))
    want = oracle.gemm_f64(A, B, ta, tb)
    # the output between guard elements: nothing outside it may be written
    buf = torch.full((M * N + 16,), 7.0, dtype=BT, device="cuda")
    C = buf[8:8 + M * N].view(M, N)
    if accumulate:
        C0 = bf16_round(g.standard_normal((M, N)))
        C.copy_(to_dev(C0, torch, BT))
        want = want + C0
    ffk.gemm(to_dev(A, torch, BT), to_dev(B, torch, BT), C, ta, tb, accumulate=accumulate)
    # exact products, fp32 accumulation, one bf16 rounding at the store
    assert_close(to_np(C), want, 2.0 ** -8, "C")
    assert bool((buf[:8] == 7.0).all()) and bool((buf[8 + M * N:] == 7.0).all())


@pytest.mark.parametrize("ta,tb", KINDS)
@pytest.mark.parametrize("variant", [64, 65, 70, 128, 256, 264])
@pytest.mark.parametrize("mnk", ALIGNED)
def test_pipelined_tiles_with_ragged_edges(ffk, oracle, ta, tb, variant, mnk):
    print("gemm edges", mnk, "ta", ta, "tb", tb, "tile", variant, flush=True)
    ffk.set_option(ffk.OPTION_GEMM_VARIANT, variant)
    try:
        product(ffk, oracle, mnk, ta, tb, accumulate=mnk[0] % 16 == 0)
    finally:
        ffk.set_option(ffk.OPTION_GEMM_VARIANT, 0)


@pytest.mark.parametrize("ta,tb", KINDS)
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("mnk", ANY)
def test_operands_of_any_alignment(ffk, oracle, ta, tb, accumulate, mnk):
    print("gemm any alignment", mnk, "ta", ta, "tb", tb, flush=True)
    product(ffk, oracle, mnk, ta, tb, accumulate)


@pytest.mark.parametrize("act", [-1, 0])
@pytest.mark.parametrize("shape", [(591, 768, 1001), (1379, 200, 776), (200, 72, 5003)])
def test_linear_bf16_ragged(ffk, oracle, shape, act):
    """Token counts and output widths that are no multiple of anything: forward with bias and
    activation, the three gradients."""
    batch, in_dim, out_dim = shape
    print("linear bf16 ragged", shape, "act", act, flush=True)
    g = rng(batch + in_dim)
    x = bf16_round(g.standard_normal((batch, in_dim)))
    w = bf16_round(g.standard_normal((out_dim, in_dim)) * 0.05)
    b = bf16_round(g.standard_normal((out_dim,)) * 0.05)
    dy = bf16_round(g.standard_normal((batch, out_dim)))
    xd, wd, bd, dyd = (to_dev(a, torch, BT) for a in (x, w, b, dy))
    y = ffk.linear_forward(xd, wd, bd, activation=act)
    assert_close(to_np(y), bf16_round(oracle.linear_forward(x, w, b, activation=act)), 2e-2, "y")
    dx_ref, dw_ref, db_ref = oracle.linear_backward(to_np(y), dy, x, w, activation=act)
    dx, dw, db = torch.zeros_like(xd), torch.zeros_like(wd), torch.zeros_like(bd)
    ffk.linear_backward(y, dyd, xd, wd, dx, dw, db, activation=act)
    for got, want, name in ((dx, dx_ref, "dx"), (dw, dw_ref, "dw"), (db, db_ref, "db")):
        assert_close(to_np(got), want, 2e-2, name)


def test_values_next_to_the_edge_stay_out(ffk):
    """Infinities in the rows and columns right behind a view's edge must not reach the result
    (0 * inf would be a NaN): operands that are corners of larger tensors are not offered by the
    entry point, so the neighbours of a dense operand are other allocations; what can be met are the
    operand's own next rows, read past a ragged K."""
    M, N, K = 72, 136, 72
    A, B = torch.ones((M, K), device="cuda", dtype=BT), torch.ones((N, K), device="cuda", dtype=BT)
    A[5, 0] = float("inf")  # follows row 4's last element in memory
    for variant in (1, 64, 128, 256):
        ffk.set_option(ffk.OPTION_GEMM_VARIANT, variant)
        try:
            C = torch.empty((M, N), device="cuda", dtype=BT)
            ffk.gemm(A, B, C, False, True)
        finally:
            ffk.set_option(ffk.OPTION_GEMM_VARIANT, 0)
        rows = torch.isinf(C).any(1)
        assert bool(rows[5]) and int(rows.sum()) == 1 and not bool(torch.isnan(C).any())
        assert bool((C[torch.arange(M, device="cuda") != 5] == K).all())


# fp32: lengths that are no multiple of four around the 64 and 128 tiles, and reductions of thousands
# over few outputs (sixteen waves a tile)
F32_ANY = [(130, 129, 33), (257, 1001, 65), (63, 300, 7), (1100, 2051, 70)]
F32_DEEP = [(25, 100, 5003), (1, 17, 2048), (250, 500, 2051), (16, 16, 4096)]


@pytest.mark.parametrize("ta,tb", KINDS)
@pytest.mark.parametrize("mnk", F32_ANY + F32_DEEP)
def test_gemm_fp32_any_lengths(ffk, oracle, ta, tb, mnk):
    M, N, K = mnk
    print("gemm fp32 any lengths", mnk, "ta", ta, "tb", tb, flush=True)
    assert ffk.gemm_kernel_name(ffk.FLOAT, ta, tb, M, N, K).startswith(
        "gemm_f32_deep" if mnk in F32_DEEP else "gemm_f32_tiled" if M * N >= 128 * 128 else "gemm_f32_kernel")
    g = rng(M * 7 + N * 3 + K)
    A = g.standard_normal((K, M) if ta else (M, K)).astype(np.float32)
    B = g.standard_normal((N, K) if tb else (K, N)).astype(np.float32)
    want = oracle.gemm_f64(A, B, ta, tb)
    buf = torch.full((M * N + 16,), 7.0, device="cuda")
    C = buf[8:8 + M * N].view(M, N)
    ffk.gemm(to_dev(A, torch), to_dev(B, torch), C, ta, tb)
    assert_close(to_np(C), want, 1e-5, "C")
    ffk.gemm(to_dev(A, torch), to_dev(B, torch), C, ta, tb, accumulate=True)
    assert_close(to_np(C), 2 * want, 1e-5, "C accumulate")
    assert bool((buf[:8] == 7.0).all()) and bool((buf[8 + M * N:] == 7.0).all())


# one per tile and wave count of the one-launch Linear kernels, sizes off every multiple of theirs
@pytest.mark.parametrize("shape", [(17, 33, 15), (3, 130, 77), (513, 41, 59), (1025, 65, 99), (601, 530, 501), (1030, 499, 510),
                                   (31, 1000, 5001)])
@pytest.mark.parametrize("act", [-1, 0, 2])
def test_linear_fp32_small_tiles(ffk, oracle, shape, act):
    batch, in_dim, out_dim = shape
    print("linear fp32 small", shape, "act", act, flush=True)
    g = rng(batch)
    x = g.uniform(-1, 1, (batch, in_dim)).astype(np.float32)
    w = (g.standard_normal((out_dim, in_dim)) * 0.2).astype(np.float32)
    b = (g.standard_normal((out_dim,)) * 0.2).astype(np.float32)
    dy = g.standard_normal((batch, out_dim)).astype(np.float32)
    y_ref = oracle.linear_forward(x, w, b, activation=act)
    xd, wd, bd, dyd = (to_dev(a, torch) for a in (x, w, b, dy))
    y = ffk.linear_forward(xd, wd, bd, activation=act)
    assert_close(to_np(y), y_ref, 1e-5, "y")
    dx_ref, dw_ref, db_ref = oracle.linear_backward(y_ref, dy, x, w, activation=act)
    got = [torch.full_like(t, 0.5) for t in (xd, wd, bd)]
    ffk.linear_backward(to_dev(y_ref, torch), dyd, xd, wd, *got, activation=act, accumulate=True)
    for t, want, name in zip(got, (dx_ref, dw_ref, db_ref), ("dx", "dw", "db")):
        assert_close(to_np(t), want + 0.5, 1e-5, name)
