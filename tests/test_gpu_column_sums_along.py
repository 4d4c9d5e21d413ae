"""An encoder layer's bias and LayerNorm gradients, added up by workgroups of the weight gradients' launch: the bits
of a launch of their own on every tile of that launch, whose workgroups have 256 or 512 threads."""
import numpy as np
import pytest

from layer_oracle import make_params
from test_gpu_encoder_layer import run_device
from util import bf16_round, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,seq,d_model,heads,d_ff", [
    (1, 17, 64, 2, 128),      # 32 x 32 tiles, one partial sum a column
    (5, 419, 160, 2, 640),    # 64 x 64 deep, columns that are no whole 32
    (5, 420, 320, 5, 1280),   # 64 x 64
    (7, 197, 768, 12, 3072),  # 128 x 128 that begin early
    (8, 512, 1024, 16, 4096),  # 256 x 256, 128 partial sums a column and more
])
@pytest.mark.parametrize("overwrite", [False, True])
def test_column_sums_beside_the_weight_gradients(ffk, batch, seq, d_model, heads, d_ff, overwrite):
    cfg = dict(batch=batch, seq=seq, d_model=d_model, heads=heads, d_ff=d_ff, p=0.1, seed=3, eps=1e-5,
               scale=0.125, causal=False, pre_ln=True, gelu=False)
    print(cfg, overwrite, flush=True)
    g = rng(seq + d_model)
    params = make_params(g, cfg, bf16_round)
    x, dy = (bf16_round(g.standard_normal((batch, seq, d_model))) for _ in range(2))
    _, _, along = run_device(ffk, cfg, params, x, dy, overwrite)
    ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 1)
    try:
        _, _, alone = run_device(ffk, cfg, params, x, dy, overwrite)
    finally:
        ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 0)
    for k in alone:
        assert np.abs(alone[k]).max() > 0
        if k not in ("attn_weight", "w1", "w2"):
            assert np.array_equal(along[k], alone[k]), k
        else:
            # the products of that launch, on tiles that may add up in another order: two roundings to bf16, of at most
            # 2^-9 of each element, and the fp32 sums' own differences far below that
            a, b = along[k].astype(np.float64), alone[k].astype(np.float64)
            assert np.linalg.norm(a - b) <= 2.0 ** -8 * np.linalg.norm(b), k
