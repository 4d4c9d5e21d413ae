"""fp32 MultiHeadAttention backward with room for dS in its reserve space (dQ is then one product of it), with room for a
part of the heads at a time, and without: the same gradients, from reserve space that holds NaN where nothing was written."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def backward(ffk, desc, x, kv, w, dout, room):
    own = kv is x
    reserve = torch.full((room,), 255, dtype=torch.uint8, device="cuda")
    ffk.mha_forward(desc, x, kv, kv, w, reserve)
    dx, dw = torch.empty_like(x), torch.zeros_like(w)
    dk, dv = (None, None) if own else (torch.empty_like(kv), torch.empty_like(kv))
    ffk.mha_backward(desc, x, dx, kv, dk, kv, dv, w, dw, dout, reserve, accumulate=ffk.MHA_OVERWRITE_WEIGHT_GRAD)
    return [t for t in (dx, dk, dv, dw) if t is not None]


@pytest.mark.parametrize("D,Dv", [(32, 32), (20, 32), (64, 64), (80, 80), (128, 128), (256, 256), (132, 256)])
@pytest.mark.parametrize("causal", [False, True])
def test_backward_with_and_without_room_for_scores(ffk, D, Dv, causal):
    # (batch, heads, queries, keys): one row; edges of the 32-row tiles; few workgroups; many of them
    for B, H, Sq, Sk in [(1, 1, 1, 1), (1, 2, 33, 31), (2, 3, 97, 130), (1, 2, 129, 64), (3, 4, 305, 305), (2, 64, 160, 160)]:
        if causal and Sq > Sk:
            Sk = Sq
        E = 64
        print("mha fp32", (D, Dv), (B, H, Sq, Sk), "causal", causal, flush=True)
        desc = ffk.mha_desc(B, H, E, E, E, D, D, Dv, E, Sq, Sk, D ** -0.5, causal)
        gen = torch.Generator(device="cuda").manual_seed(Sq + D)
        mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
        x = mk(B, Sq, E)
        kv = x if Sq == Sk else mk(B, Sk, E)
        w = mk(ffk.lib().ffk_mha_weight_elements(desc)) * 0.2
        dout = mk(B, Sq, E)
        full = ffk.mha_reserve(desc, ffk.FLOAT).numel()
        scores = 4 * B * H * Sq * ((Sk + 31) // 32 * 32)
        want = backward(ffk, desc, x, kv, w, dout, full - scores)
        for room in (full, full - 16):  # the second: a part too small for a launch of its own, as without room
            for name, a, b in zip(("dx", "dk", "dv", "dw"), backward(ffk, desc, x, kv, w, dout, room), want):
                # two orders of the same fp32 sums
                assert float((a - b).double().norm() / b.double().norm()) <= 8 * 2.0 ** -24 * max(Sq, Sk) ** 0.5, (name, room)
        with pytest.raises(ffk.FFKError, match="reserve space"):
            backward(ffk, desc, x, kv, w, dout, full - scores - 256)


def test_backward_with_room_for_half_of_the_heads(ffk):
    """1024 heads, 512 at a time: two launches of each kernel."""
    B, H, S, D, E = 8, 128, 128, 32, 32
    desc = ffk.mha_desc(B, H, E, E, E, D, D, D, E, S, S, D ** -0.5, True)
    print("mha fp32, half of the heads at a time", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(1)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    x, w, dout = mk(B, S, E), mk(ffk.lib().ffk_mha_weight_elements(desc)) * 0.2, mk(B, S, E)
    full, scores = ffk.mha_reserve(desc, ffk.FLOAT).numel(), 4 * B * H * S * S
    want = backward(ffk, desc, x, x, w, dout, full)
    for a, b in zip(backward(ffk, desc, x, x, w, dout, full - scores // 2), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("D", [32, 64, 80, 128, 132, 256])
@pytest.mark.parametrize("causal", [False, True])
def test_backward_with_room_for_a_part_of_the_heads(ffk, D, causal):
    """700 heads of 128 or 121 rows, 520 at a time and then the 180 left, whose products of dS are shared out among more workgroups."""
    B, H, S, E = 10, 70, 128 if D > 128 else 121, 16
    print("mha fp32, 520 and 180 of 700 heads", D, causal, flush=True)
    desc = ffk.mha_desc(B, H, E, E, E, D, D, D, E, S, S, D ** -0.5, causal)
    gen = torch.Generator(device="cuda").manual_seed(D)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    x, w, dout = mk(B, S, E), mk(ffk.lib().ffk_mha_weight_elements(desc)) * 0.2, mk(B, S, E)
    full, one = ffk.mha_reserve(desc, ffk.FLOAT).numel(), 4 * S * 128
    assert ffk.lib().ffk_mha_backward_workspace_bytes(ctypes.byref(desc), ffk.FLOAT) == 700 * one
    want = backward(ffk, desc, x, x, w, dout, full)
    for a, b in zip(backward(ffk, desc, x, x, w, dout, full - 179 * one - 16), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("D,causal", [(64, True), (256, False)])
def test_backward_with_room_that_layers_share(ffk, D, causal):
    """dS in memory of its own: the bits of dS behind what is kept; lent unaligned, the bits without any."""
    B, H, S, E = 2, 3, 97, 64
    print("mha fp32, shared workspace", D, flush=True)
    desc = ffk.mha_desc(B, H, E, E, E, D, D, D, E, S, S, D ** -0.5, causal)
    gen = torch.Generator(device="cuda").manual_seed(D)
    mk = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    x, w, dout = mk(B, S, E), mk(ffk.lib().ffk_mha_weight_elements(desc)) * 0.2, mk(B, S, E)
    reserve, ws = ffk.mha_reserve(desc, ffk.FLOAT, backward_scratch=False), ffk.mha_backward_workspace(desc, ffk.FLOAT)
    full = ffk.mha_reserve(desc, ffk.FLOAT).numel()
    assert reserve.numel() + ws.numel() == full and ws.numel() == 4 * B * H * S * 128
    ffk.mha_forward(desc, x, x, x, w, reserve)
    for lent, same_as in ((ws, full), (ws[4:], reserve.numel())):
        dx, dw = torch.empty_like(x), torch.zeros_like(w)
        ffk.mha_backward(desc, x, dx, x, None, x, None, w, dw, dout, reserve, ffk.MHA_OVERWRITE_WEIGHT_GRAD, workspace=lent)
        for a, b in zip((dx, dw), backward(ffk, desc, x, x, w, dout, same_as)):
            assert torch.equal(a, b)
