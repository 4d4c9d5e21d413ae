"""An encoder layer's weight gradients, taken together, over long reductions: on every tile of the group's launch the
gradients of the products taken one by one."""
import numpy as np
import pytest

from layer_oracle import make_params
from test_gpu_encoder_layer import run_device
from util import assert_close, bf16_round, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,seq,d_model,heads,d_ff", [
    (5, 420, 64, 2, 128), (9, 233, 64, 2, 256),      # 32 x 32 tiles, a round and more
    (5, 419, 160, 2, 640), (4, 520, 256, 4, 1024),   # 64 x 64 deep, a ragged and a whole reduction
    (5, 420, 320, 5, 1280), (6, 350, 512, 8, 1024),  # 64 x 64, 128 x 128
])
@pytest.mark.parametrize("overwrite", [False, True])
def test_gradients_together_and_one_by_one(ffk, batch, seq, d_model, heads, d_ff, overwrite):
    cfg = dict(batch=batch, seq=seq, d_model=d_model, heads=heads, d_ff=d_ff, p=0.0, seed=1, eps=1e-5,
               scale=0.125, causal=False, pre_ln=True, gelu=True)
    print(cfg, flush=True)
    g = rng(seq)
    params = make_params(g, cfg, bf16_round)
    x, dy = (bf16_round(g.standard_normal((batch, seq, d_model))) for _ in range(2))
    _, dx, together = run_device(ffk, cfg, params, x, dy, overwrite)
    ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 1)
    try:
        _, dx1, alone = run_device(ffk, cfg, params, x, dy, overwrite)
    finally:
        ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 0)
    assert np.array_equal(dx, dx1)  # the same operands
    for k in ("attn_weight", "w1", "w2"):
        assert np.abs(alone[k]).max() > 0
        # float32 sums of the same products in another order, each rounded to bfloat16 once
        assert_close(together[k], alone[k], 2.0 ** -8, k)
