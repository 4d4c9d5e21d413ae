"""Products, attention and updates whose kernels are chosen for few elements: fp32 products on register-fed tiles,
bf16 products of unaligned rows with a wave to an output, and the fp32 attention backward on both sides of the
size where two waves stop sharing their rows.  References are float64 on the CPU."""
import pytest
import torch

from util import assert_close, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("mnk", [(138, 640, 640), (129, 130, 256), (1023, 255, 1024), (17, 15000, 259), (799, 801, 1021)])
def test_gemm_fp32_small_tiles(ffk, ta, tb, mnk):
    M, N, K = mnk
    print("gemm fp32 small", mnk, ta, tb, flush=True)
    assert ffk.gemm_kernel_name(ffk.FLOAT, ta, tb, M, N, K).startswith("gemm_f32_small")
    gen = torch.Generator().manual_seed(M + N + K)
    A, B = torch.randn((K, M) if ta else (M, K), generator=gen), torch.randn((N, K) if tb else (K, N), generator=gen)
    want = to_np((A.t() if ta else A).double() @ (B.t() if tb else B).double())
    buf = torch.full((M * N + 16,), 7.0, device="cuda")
    C = buf[8:8 + M * N].view(M, N)
    ffk.gemm(A.cuda(), B.cuda(), C, ta, tb)
    assert_close(to_np(C), want, 1e-5, "C")
    ffk.gemm(A.cuda(), B.cuda(), C, ta, tb, accumulate=True)
    assert_close(to_np(C), 2 * want, 1e-5, "C accumulate")
    assert bool((buf[:8] == 7.0).all()) and bool((buf[8 + M * N:] == 7.0).all())


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("mnk", [(17, 43, 841), (1, 1, 64), (51, 131, 251), (43, 841, 17), (9, 7, 63), (3, 5, 20001), (52, 37, 1907), (129, 127, 513)])
def test_gemm_bf16_few_outputs(ffk, ta, tb, mnk):
    M, N, K = mnk
    print("gemm bf16 few outputs", mnk, ta, tb, flush=True)
    gen = torch.Generator().manual_seed(M + N + K)
    A = torch.randn((K, M) if ta else (M, K), generator=gen).bfloat16()
    B = torch.randn((N, K) if tb else (K, N), generator=gen).bfloat16()
    want = to_np((A.t() if ta else A).double() @ (B.t() if tb else B).double())
    C = torch.empty((M, N), device="cuda", dtype=torch.bfloat16)
    ffk.gemm(A.cuda(), B.cuda(), C, ta, tb)
    # one rounding to bf16 of an fp32 sum: half a unit in the last of 8 bits
    assert_close(to_np(C.float()), want, 2.0 ** -8, "C")


@pytest.mark.parametrize("shape", [(37, 61, 9001), (5, 17, 4097), (128, 45, 20001), (300, 40, 2048)])
def test_linear_fp32_backward_split_reduction(ffk, shape):
    """The input gradient's reduction over thousands of outputs, split over workgroups."""
    B, I, O = shape
    gen = torch.Generator().manual_seed(B + I + O)
    x, w, dy, y = (torch.randn(s, generator=gen) for s in ((B, I), (O, I), (B, O), (B, O)))
    dx, dw, db = (torch.full(s, 3.0, device="cuda") for s in ((B, I), (O, I), (O,)))
    ffk.linear_backward(y.cuda(), dy.cuda(), x.cuda(), w.cuda(), dx, dw, db, activation=ffk.ACT_NONE)
    for t, want, name in ((dx, dy.double() @ w.double(), "dx"), (dw, dy.double().t() @ x.double(), "dw"), (db, dy.double().sum(0), "db")):
        assert_close(to_np(t), to_np(want), 1e-5, name)


@pytest.mark.parametrize("shape", [(1, 2, 1, 9, 64), (1, 3, 65, 33, 128), (2, 8, 138, 58, 80), (16, 16, 70, 70, 64),
                                   (16, 16, 40, 130, 128), (8, 17, 130, 100, 72), (16, 32, 20, 20, 32), (1, 2, 97, 64, 256)])
@pytest.mark.parametrize("causal", [False, True])
def test_attention_fp32_backward_both_forms(ffk, shape, causal):
    B, H, Sq, Skv, D = shape
    # causal with Sq != Skv: key j is visible to query i iff j <= i
    print("attention fp32", shape, causal, flush=True)
    gen = torch.Generator().manual_seed(Sq + D)
    q, k, v, do = (torch.randn((B, s, H, D), generator=gen) for s in (Sq, Skv, Skv, Sq))
    scale = D ** -0.5
    qt, kt, vt, dot = (t.double().transpose(1, 2).contiguous() for t in (q, k, v, do))
    s = (qt @ kt.transpose(2, 3).contiguous()) * scale
    if causal:
        s = s.masked_fill(torch.ones(Sq, Skv, dtype=torch.bool).triu(1), float("-inf"))
    p = s.softmax(-1)
    o_ref = p @ vt
    dp = dot @ vt.transpose(2, 3).contiguous()
    ds = p * (dp - (dot * o_ref).sum(-1, keepdim=True)) * scale
    want = (ds @ kt, ds.transpose(2, 3).contiguous() @ qt, p.transpose(2, 3).contiguous() @ dot)
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    o, lse = ffk.attention_forward(qd, kd, vd, scale, causal)
    assert_close(to_np(o), to_np(o_ref.transpose(1, 2).contiguous()), 1e-5, "O")
    got = ffk.attention_backward(qd, kd, vd, o, dod, lse, scale, causal)
    # where the only query sees one key, of dQ and dK nothing is left but the rounding of dP - delta: 1e-5 of
    # these two, times the other factor
    rest = 1e-5 * float(dp.abs().max()) * scale * max(float(t.abs().max()) for t in (qt, kt)) if causal and Sq == 1 else 0.0
    for t, w, name in zip(got, want, ("dQ", "dK", "dV")):
        if rest > 0 and name != "dV":
            assert float(t.abs().max()) <= rest, name
        else:
            assert_close(to_np(t), to_np(w.transpose(1, 2).contiguous()), 1e-5, name)


@pytest.mark.parametrize("n,dtype,copy", [(8388609, torch.float32, True), (8389631, torch.float32, True),
                                          (20971520, torch.float32, False), (20972543, torch.float32, False),
                                          (33554433, torch.bfloat16, False)])
def test_adam_past_the_caches(ffk, oracle, n, dtype, copy):
    """Parameters from where the update bypasses the caches on, with a last workgroup of few, on both sides of the
    sizes from which a thread takes two vectors again."""
    gen = torch.Generator().manual_seed(n)
    w0, grad, m0 = (torch.randn(n, generator=gen) for _ in range(3))
    grad = grad.to(dtype)
    v0 = torch.rand(n, generator=gen)
    args = dict(alpha_t=1e-2, beta1=0.9, beta2=0.99, weight_decay=0.05, epsilon=1e-6)
    want = oracle.adam_update(w0.numpy().copy(), grad.float().numpy().copy(), m0.numpy().copy(), v0.numpy().copy(), **args)
    w, m, v = w0.cuda(), m0.cuda(), v0.cuda()
    low = torch.empty(n, device="cuda", dtype=torch.bfloat16) if copy else None
    ffk.adam_update(w, grad.cuda(), m, v, weight_lowp=low, **args)
    for got, ref in zip((w, m, v), want):
        assert torch.equal(got.cpu(), torch.from_numpy(ref))
    assert low is None or torch.equal(low, w.to(torch.bfloat16))
