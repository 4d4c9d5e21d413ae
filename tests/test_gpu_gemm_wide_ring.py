"""The bf16 product on tiles of one wave per SIMD, whose k-tiles pass through a ring of five panels: the bits of the
128 x 128 tiles, on 32 x 32 matrix instructions, over reductions of one k-tile and up to past the ring's second round."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def product(ffk, variant, a, b, ta, tb, c0):
    c = c0.clone()
    ffk.set_option(ffk.OPTION_GEMM_VARIANT, variant)
    try:
        ffk.gemm(a, b, c, trans_a=ta, trans_b=tb, accumulate=bool(c0.abs().sum() > 0))
    finally:
        ffk.set_option(ffk.OPTION_GEMM_VARIANT, 0)
    return c


@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 384, 704])
@pytest.mark.parametrize("accumulate", [False, True])
def test_ring_of_panels(ffk, ta, tb, K, accumulate):
    M, N = 512, 256
    print("wide tile", (M, N, K), ta, tb, accumulate, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(K)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()  # noqa: E731
    a, b = mk(*((K, M) if ta else (M, K))), mk(*((N, K) if tb else (K, N)))
    c0 = mk(M, N) if accumulate else torch.zeros(M, N, device="cuda", dtype=torch.bfloat16)
    assert torch.equal(product(ffk, 264, a, b, ta, tb, c0), product(ffk, 128, a, b, ta, tb, c0))


@pytest.mark.parametrize("K", [1024, 1088, 1216])
def test_ring_of_panels_192_columns(ffk, K):
    M, N = 256, 384
    print("wide tile of 192 columns", (M, N, K), flush=True)
    gen = torch.Generator(device="cuda").manual_seed(K)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()  # noqa: E731
    a, b, c0 = mk(M, K), mk(N, K), torch.zeros(M, N, device="cuda", dtype=torch.bfloat16)
    assert torch.equal(product(ffk, 192, a, b, False, True, c0), product(ffk, 128, a, b, False, True, c0))
