"""fp32 attention where waves, or pairs of them, share out the streamed rows: sequences around a step of each form,
rows that only some waves see, two head sizes, the causal mask, and enough heads that nothing is shared."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(32, 32), (64, 64), (40, 64), (80, 80), (128, 128), (128, 36)])
@pytest.mark.parametrize("causal", [False, True])
def test_attention_fp32_of_any_split(ffk, sizes, causal):
    D, Dv = sizes
    for B, H, Sq, Skv in [(1, 1, 1, 1), (1, 2, 33, 31), (1, 2, 129, 65), (2, 3, 97, 301), (1, 2, 270, 530), (2, 16, 150, 200), (2, 33, 260, 140)]:
        if causal and Sq > Skv:
            Skv = Sq
        print("attention fp32", sizes, (B, H, Sq, Skv), "causal", causal, flush=True)
        gen = torch.Generator(device="cuda").manual_seed(Sq + D)
        mk = lambda s, d: torch.randn(B, s, H, d, device="cuda", generator=gen)  # noqa: E731
        q, k, v, g = mk(Sq, D), mk(Skv, D), mk(Skv, Dv), mk(Sq, Dv)
        scale = D ** -0.5
        o, lse = ffk.attention_forward(q, k, v, scale, causal)
        dq, dk, dv = ffk.attention_backward(q, k, v, o, g, lse, scale, causal)
        Q, K, V, G = (t.double().transpose(1, 2).contiguous() for t in (q, k, v, g))
        s = Q @ K.transpose(-1, -2) * scale
        if causal:
            s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), float("-inf"))
        p = torch.softmax(s, -1)
        O = p @ V
        # a score is off by the roundings of its sum, a probability by as much relatively; sums over keys add theirs
        u = 2.0 ** -24 * (8 * (D + Skv) ** 0.5 + 64)
        got = lambda t: t.double().transpose(1, 2)  # noqa: E731
        eo = u * (p @ V.abs()) + 1e-12
        assert bool(((got(o) - O).abs() <= eo).all()), float(((got(o) - O).abs() / eo).max())
        dp = G @ V.transpose(-1, -2)
        ds = p * (dp - (G * O).sum(-1, keepdim=True)) * scale
        size = p * scale * (G.abs() @ V.abs().transpose(-1, -2) + (G * O).abs().sum(-1, keepdim=True) + (G.abs() * (p @ V.abs())).sum(-1, keepdim=True))
        pt, st, dt = p.transpose(-1, -2), size.transpose(-1, -2), ds.transpose(-1, -2)
        for name, x, want, bound in (("dv", dv, pt @ G, pt @ G.abs()), ("dq", dq, ds @ K, size @ K.abs()), ("dk", dk, dt @ Q, st @ Q.abs())):
            e = (got(x) - want).abs()
            assert bool((e <= u * bound + 1e-12).all()), (name, float((e / (u * bound + 1e-12)).max()))
