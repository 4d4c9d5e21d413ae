"""LayerNorm and Softmax where a row's lanes, and its last vector, can go wrong: lengths around whole vectors
and around the groups of 16, 32 and 64 lanes, row counts around what a workgroup holds, any alignment."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LENGTHS = [1, 3, 7, 9, 63, 64, 65, 127, 128, 129, 136, 255, 256, 257, 511, 513, 520, 1023, 1025, 2049, 4095, 8190]


def placed(x, shift):
    """A copy of x that begins `shift` elements behind a 16-byte boundary, and what surrounds it."""
    room = torch.full((x.numel() + 32,), 5.0, device="cuda", dtype=x.dtype)
    view = room[8 + shift:8 + shift + x.numel()].view(x.shape)
    view.copy_(x)
    return view, room


def untouched(room, shift, n):
    return bool((room[:8 + shift] == 5.0).all()) and bool((room[8 + shift + n:] == 5.0).all())


def close(got, want, magnitude, n, dtype):
    """A result of sums over n float32 terms, stored as dtype: each sum is at most (log2 n + 16) roundings off
    its terms' magnitudes, a result a few such; storing rounds it once more, by 2^-9 in bfloat16."""
    store = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    bound = 8 * (n.bit_length() + 16) * 2.0 ** -24 * magnitude + store * want.abs()
    err = (got.double() - want).abs()
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,shift", [(1, 1), (37, 0), (37, 3), (1100, 1)])
def test_rows_of_any_length(ffk, dtype, rows, shift):
    gen = torch.Generator(device="cuda").manual_seed(rows + shift)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    for N in LENGTHS:
        print("rows", rows, "of", N, dtype, "shift", shift, flush=True)
        x, dy, dx0 = ((1.5 * rand(rows, N) + 0.3).to(dtype) for _ in range(3))
        gamma, beta = (1 + 0.1 * rand(N)).to(dtype), (0.1 * rand(N)).to(dtype)
        xd, dyd, gd, bd = (placed(t, shift)[0] for t in (x, dy, gamma, beta))
        y, mean, rstd = ffk.layer_norm_forward(xd, gd, bd, 1e-5)
        X, DY, G, B = (t.double() for t in (x, dy, gamma, beta))
        mu = X.mean(1, keepdim=True)
        rs = 1 / torch.sqrt(((X - mu) ** 2).mean(1, keepdim=True) + 1e-5)
        xh = (X - mu) * rs
        # the error of x - mean, relative to the row's largest element, is scaled by rstd and gamma
        big = X.abs().amax(1, keepdim=True) * rs
        close(mean[:, None], mu, X.abs().amax(1, keepdim=True), N, torch.float32)
        close(rstd[:, None], rs, rs * (1 + big ** 2), N, torch.float32)
        close(y, xh * G + B, (1 + big) ** 2 * G.abs() + B.abs(), N, dtype)
        D = DY * G
        want = rs * (D - D.mean(1, keepdim=True) - xh * (D * xh).mean(1, keepdim=True))
        size = rs * D.abs().amax(1, keepdim=True) * (1 + big) ** 3
        for acc in (False, True):
            dx, room = placed(dx0, shift)
            dg, db = torch.zeros_like(gamma), torch.zeros_like(beta)
            ffk.layer_norm_backward(dyd, xd, mean, rstd, gd, dx, dg, db, accumulate=acc)
            base = dx0.double() if acc else torch.zeros_like(X)
            close(dx, want + base, size + base.abs(), N, dtype)
            assert untouched(room, shift, rows * N)
            close(dg, (DY * xh).sum(0), (DY.abs() * (1 + big) ** 2).sum(0), rows, dtype)
            close(db, DY.sum(0), DY.abs().sum(0), rows, dtype)
        # softmax: e^(x - max) <= 1 to a few float32 roundings of x - max
        p = ffk.softmax_forward(xd, rows, N, 1)
        P = torch.softmax(X, 1)
        close(p, P, P * (2 + (X.amax(1, keepdim=True) - X)), N, dtype)
        DP = p.double()
        pd, _ = placed(p, shift)
        ds = ffk.softmax_backward(pd, dyd, rows, N, 1)
        dot = (DP * DY).sum(1, keepdim=True)
        close(ds, DP * (DY - dot), DP * (DY.abs() + (DP * DY.abs()).sum(1, keepdim=True)), N, dtype)
        if shift and N % 8 == 0:  # the same lanes hold the same elements wherever the rows lie
            assert torch.equal(y, ffk.layer_norm_forward(x, gamma, beta, 1e-5)[0])
            assert torch.equal(p, ffk.softmax_forward(x, rows, N, 1))
