"""fp32 products whose tiles' waves split the reduction: two and four groups, reductions around whole k-tiles and
shorter than a group's share, ragged tiles, every operand order, aligned and not."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("mnk", [
    (1024, 768, 1056), (1021, 769, 1025), (960, 1020, 1316), (1000, 1000, 256), (1000, 700, 289),  # 64 x 64, two groups
    (1024, 768, 2048), (1027, 641, 2177), (700, 1000, 2303),                                      # four
    (2048, 768, 257), (1090, 1020, 1100), (2041, 515, 480), (1100, 1024, 4100)])                  # 128 x 64, two
def test_groups(ffk, ta, tb, mnk):
    M, N, K = mnk
    name = ffk.gemm_kernel_name(ffk.FLOAT, ta, tb, M, N, K)
    print(mnk, ta, tb, name, flush=True)
    assert name.startswith("gemm_f32_tiled_kernel") and name.endswith((",2>", ",4>"))
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    rand = lambda *s: torch.randn(s, device="cuda", generator=gen)  # noqa: E731
    a, b, bias = rand(K, M) if ta else rand(M, K), rand(N, K) if tb else rand(K, N), rand(N)
    A, B = (a.t() if ta else a).double(), (b.t() if tb else b).double()
    want, size = A @ B, A.abs() @ B.abs()
    # a float32 sum of K products in any order: K roundings at most, in fact their root
    bound = 4 * K ** 0.5 * 2.0 ** -24 * size
    room = torch.full((M * N + 64,), 7.0, device="cuda")
    c = room[32:32 + M * N].view(M, N)
    ffk.gemm(a, b, c, ta, tb)
    assert bool(((c.double() - want).abs() <= bound).all())
    ffk.gemm(a, b, c, ta, tb, accumulate=True)
    assert bool(((c.double() - 2 * want).abs() <= 2 * bound + 2.0 ** -22 * want.abs()).all())
    assert bool((room[:32] == 7.0).all()) and bool((room[32 + M * N:] == 7.0).all())
    if not ta and tb:
        y = ffk.linear_forward(a, b, bias, activation=ffk.ACT_RELU)
        assert bool(((y.double() - (want + bias.double()).clamp(min=0)).abs() <= bound + 2.0 ** -22 * (want.abs() + bias.abs())).all())
