"""bf16 attention where the waves of a workgroup share out the streamed rows, and of head sizes between the padded
ones: sequences around a step of each form, rows that only some waves see, two head sizes, the causal mask."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# head sizes of Q and K, of V; the last two run the tuned kernels' sizes with so few workgroups that they do not
SIZES = [(8, 8), (32, 32), (24, 40), (64, 48), (80, 80), (96, 72), (104, 128), (256, 256), (136, 200), (64, 64), (128, 128)]
# batch, heads, queries, keys: one workgroup, some, and more than the chip has CUs of each form
SHAPES = [(1, 1, 1, 1), (1, 2, 33, 31), (1, 2, 129, 65), (2, 3, 97, 301), (1, 2, 270, 530), (2, 33, 260, 140), (3, 96, 257, 66)]


def reference(q, k, v, g, scale, causal):
    s = q @ k.transpose(-1, -2) * scale
    if causal:
        s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), float("-inf"))
    p = torch.softmax(s, -1)
    o = p @ v
    dp = g @ v.transpose(-1, -2)
    ds = p * (dp - (g * o).sum(-1, keepdim=True)) * scale
    return p, o, ds


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("causal", [False, True])
def test_attention_of_any_split(ffk, sizes, causal):
    D, Dv = sizes
    u = 2.0 ** -9  # a rounding to bfloat16
    for B, H, Sq, Skv in SHAPES:
        if causal and Sq > Skv:
            Skv = Sq
        print("attention", sizes, (B, H, Sq, Skv), "causal", causal, flush=True)
        gen = torch.Generator(device="cuda").manual_seed(Sq + D)
        mk = lambda s, d: torch.randn(B, s, H, d, device="cuda", generator=gen).to(torch.bfloat16)  # noqa: E731
        q, k, v, g = mk(Sq, D), mk(Skv, D), mk(Skv, Dv), mk(Sq, Dv)
        scale = D ** -0.5
        o, lse = ffk.attention_forward(q, k, v, scale, causal)
        dq, dk, dv = ffk.attention_backward(q, k, v, o, g, lse, scale, causal)
        Q, K, V, G = (t.double().transpose(1, 2).contiguous() for t in (q, k, v, g))
        p, O, ds = reference(Q, K, V, G, scale, causal)
        got = lambda t: t.double().transpose(1, 2)  # noqa: E731
        # P is rounded for the product with V, the result once more; twice that covers the sums in float32
        eo = 2 * u * (p @ V.abs() + O.abs())
        assert bool(((got(o) - O).abs() <= eo).all()), float(((got(o) - O).abs() / eo).max())
        eg = 2 * u * (p.transpose(-1, -2) @ G.abs())
        assert bool(((got(dv) - p.transpose(-1, -2) @ G).abs() <= 2 * eg).all())
        # dS is rounded for the products with K and Q; what it takes from delta inherits O's error
        eds = 2 * u * ds.abs() + p * scale * (G.abs() * eo).sum(-1, keepdim=True)
        for name, x, want, other in (("dq", dq, ds @ K, eds @ K.abs()),
                                     ("dk", dk, ds.transpose(-1, -2) @ Q, eds.transpose(-1, -2) @ Q.abs())):
            bound = other + 2 * u * want.abs() + 1e-6
            assert bool(((got(x) - want).abs() <= bound).all()), (name, float(((got(x) - want).abs() / bound).max()))
