"""Linear backward where the input gradient's reduction over the outputs is split over workgroups: partial
sums in the workspace, added up behind the product."""
import pytest
import torch

from util import assert_close, to_np

pytestmark = pytest.mark.gpu
BT = torch.bfloat16

# batch, in, out.  bf16: 128 x 128 tiles, whole and beginning early, and 256 x 256 tiles; rows of the
# gradient padded and not.  fp32: 16 x 16 tiles.
BF16 = [(130, 136, 9001), (256, 256, 8192), (700, 520, 30001), (663, 1480, 20001)]
FP32 = [(37, 61, 9001), (5, 17, 4097), (128, 45, 20001), (300, 40, 2048)]
SHAPES = [(BT, s) for s in BF16] + [(torch.float32, s) for s in FP32]


def tensors(dtype, shape):
    B, I, O = shape
    gen = torch.Generator(device="cuda").manual_seed(B + I + O)
    return [torch.randn(s, generator=gen, device="cuda").to(dtype) for s in ((B, O), (B, O), (B, I), (O, I))]


def check(got, want, dtype, what):
    """want in float64.  fp32: as every fp32 product here.  bf16: one rounding of an fp32 sum."""
    assert_close(to_np(got), want.cpu().numpy(), 1e-5 if dtype == torch.float32 else 2.0 ** -8, what)


@pytest.mark.parametrize("dtype,shape", SHAPES)
def test_bits_do_not_depend_on_the_other_gradients(ffk, dtype, shape):
    """The input gradient, whether the weight gradient is stored, added to or not asked for, and whether
    there is a bias gradient."""
    print("split reduction", dtype, shape, flush=True)
    B, I, O = shape
    y, dy, x, w = tensors(dtype, shape)

    def backward(dw, db, accumulate, act=ffk.ACT_NONE):
        dx = torch.full_like(x, 3.0)
        ffk.linear_backward(y, dy, x, w, dx, dw, db, activation=act, accumulate=accumulate)
        return dx

    dw, db = torch.full_like(w, 3.0), torch.full((O,), 3.0, device="cuda", dtype=dtype)
    dx = backward(dw, db, 0)
    check(dx, dy.double() @ w.double(), dtype, "dx")
    check(dw, dy.double().t() @ x.double(), dtype, "dw")
    check(db, dy.double().sum(0), dtype, "db")
    assert torch.equal(backward(None, db, 0), dx)
    assert torch.equal(backward(None, None, 0), dx)
    once = dw.clone()
    assert torch.equal(backward(dw, db, 2 | 4), dx)  # FFK_ACC_WEIGHT | FFK_ACC_BIAS
    assert_close(to_np(dw), 2 * to_np(once), 2.0 ** -7 if dtype == BT else 1e-5, "dw added")
    # dx added to, and an activation
    added = x.clone()
    ffk.linear_backward(y, dy, x, w, added, dw, db, accumulate=7)
    check(added, dy.double() @ w.double() + x.double(), dtype, "dx added")
    g = torch.where(y > 0, dy, torch.zeros_like(dy)).double()
    check(backward(dw, db, 0, ffk.ACT_RELU), g @ w.double(), dtype, "dx behind ReLU")


@pytest.mark.parametrize("dtype,shape", [(BT, BF16[0]), (BT, BF16[1]), (torch.float32, FP32[0])])
def test_workspace_of_every_size(ffk, dtype, shape):
    """From the least the call can do with to more than the query asks for, nothing outside of it written."""
    B, I, O = shape
    y, dy, x, w = tensors(dtype, shape)
    need = ffk.lib().ffk_linear_backward_workspace_bytes(ffk.dtype_of(x), ffk.ACT_NONE, 1, B, O)
    assert need == ffk.lib().ffk_linear_backward_workspace_bytes(ffk.dtype_of(x), ffk.ACT_NONE, 0, B, O) + \
        -(-(-(-B // 32) * O * 4) // 256) * 256  # the column sums of blocks of 32 rows
    want = dy.double() @ w.double()
    least = -(-(-(-B // 32) * O * 4) // 256) * 256
    for size in (least, least + 256, need - 256, need - 1, need, need + 1, need + 4096):
        ws = torch.full((size + 512,), 0x7f, dtype=torch.uint8, device="cuda")
        dx, dw, db = torch.full_like(x, 3.0), torch.full_like(w, 3.0), torch.full((O,), 3.0, device="cuda", dtype=dtype)
        ffk.linear_backward(y, dy, x, w, dx, dw, db, workspace=ws[256:256 + size])
        assert bool((ws[:256] == 0x7f).all()) and bool((ws[256 + size:] == 0x7f).all())
        check(dx, want, dtype, "dx with %d bytes" % size)
        check(db, dy.double().sum(0), dtype, "db with %d bytes" % size)
    ws = torch.empty((least - 256,), dtype=torch.uint8, device="cuda")
    with pytest.raises(ffk.FFKError, match="workspace"):
        ffk.linear_backward(y, dy, x, w, dx, dw, db, workspace=ws)


def test_column_sums_that_wait_in_the_workspace(ffk):
    """A bias gradient whose last step is collected, and the input gradient of the same Linear behind it with
    the same workspace: its partial sums leave the column sums alone."""
    B, I, O = 256, 256, 8192
    _, dy, x, w = tensors(BT, (B, I, O))
    need = ffk.lib().ffk_linear_backward_workspace_bytes(ffk.BF16, ffk.ACT_NONE, 1, B, O)
    ws = torch.empty((need,), dtype=torch.uint8, device="cuda")
    g, db, dx = torch.empty_like(dy), torch.zeros(O, device="cuda", dtype=BT), torch.empty_like(x)
    ffk.check(ffk.lib().ffk_column_reductions_begin())
    try:
        ffk._call.ffk_dropout_backward_bias_grad(ffk.BF16, dy, g, B, O, db, 0, ws, need, 0.0, 1, 0)
        ffk.linear_backward(None, g, x, w, dx, workspace=ws)
    finally:
        ffk.check(ffk.lib().ffk_column_reductions_end(ffk.current_stream()))
    assert torch.equal(g, dy)
    check(db, dy.double().sum(0), BT, "db")
    check(dx, dy.double() @ w.double(), BT, "dx")
