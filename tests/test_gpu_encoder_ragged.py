"""Encoder layer at token counts and widths that are no whole tiles: against the oracle at a small size,
and the fused layer against one kernel per operator where every fused form runs on ragged tiles."""
import numpy as np
import pytest
import torch

from layer_oracle import layer_forward_backward, make_params
from test_gpu_encoder_layer import run_device
from util import assert_close, bf16_round, rng

pytestmark = pytest.mark.gpu


def inputs(batch, seq, d_model, heads, d_ff, pre_ln, gelu):
    cfg = dict(batch=batch, seq=seq, d_model=d_model, heads=heads, d_ff=d_ff, p=0.1, seed=77, eps=1e-5,
               scale=0.125, causal=False, pre_ln=pre_ln, gelu=gelu)
    g = rng(batch * seq)
    params = make_params(g, cfg, bf16_round)
    for k in ("attn_weight", "w1", "w2"):
        params[k] = bf16_round(params[k] * 3)
    x = bf16_round(g.standard_normal((batch, seq, d_model)))
    return cfg, params, x, bf16_round(g.standard_normal(x.shape))


@pytest.mark.parametrize("pre_ln,gelu", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("shape", [(3, 37, 128, 2, 264), (1, 17, 160, 2, 320)])
def test_ragged_layer_against_the_oracle(ffk, oracle, shape, pre_ln, gelu):
    cfg, params, x, dy = inputs(*shape, pre_ln, gelu)
    print("ragged encoder layer", cfg, flush=True)
    y_ref, dx_ref, g_ref = layer_forward_backward(oracle, cfg, params, x, dy)
    y, dx, grads = run_device(ffk, cfg, params, x, dy)
    assert_close(y, y_ref, 2e-2, "y")
    assert_close(dx, dx_ref, 2e-2, "dx")
    for k in g_ref:
        assert_close(grads[k].reshape(g_ref[k].shape), g_ref[k], 2e-2, "grad " + k)


@pytest.mark.parametrize("pre_ln,gelu", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("shape", [(3, 37, 128, 2, 264), (7, 197, 768, 12, 3072), (8, 228, 1024, 16, 4096)])
def test_ragged_fused_layer_equals_operator_sequence(ffk, shape, pre_ln, gelu):
    """Activations, input gradient and bias / LayerNorm gradients bit for bit; the weight matrices'
    gradients, which run as one launch on a tile chosen for all of them together, to an fp32
    summation order (one rounding step of bf16 at most)."""
    cfg, params, x, dy = inputs(*shape, pre_ln, gelu)
    print("ragged fused against sequence", cfg, flush=True)
    ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 1)
    try:
        y_u, dx_u, g_u = run_device(ffk, cfg, params, x, dy)
    finally:
        ffk.set_option(ffk.OPTION_LAYER_UNFUSED, 0)
    y_f, dx_f, g_f = run_device(ffk, cfg, params, x, dy)
    assert np.array_equal(y_u, y_f) and np.array_equal(dx_u, dx_f)
    for k in g_u:
        if k in ("w1", "w2", "attn_weight"):
            assert_close(g_f[k], g_u[k], 2.0 ** -7, k)
        else:
            assert np.array_equal(g_u[k], g_f[k]), k
