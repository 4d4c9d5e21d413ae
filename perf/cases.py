"""The work that programs built on this library have it do, as cases that can be timed.

`listed()` names the cases, `draw(rng)` gives further ones of the same ranges, `prepare(case, seed)`
makes what a program has in hand before the call (tensors on the GPU, descriptors, workspaces), and
`run(state)` makes one pass through the package's entry points.  Sizes are those of the repository's
benchmark and tests, or generic ones between them.  Import with the repository root first in
sys.path: the package is the one found from there.

Kinds of work
  linear     one Linear layer, forward and backward (input, weight and bias gradients)
  encoder    one transformer encoder layer, forward and backward, BF16
  mha        one MultiHeadAttention block (projections and core), forward and backward
  rowwise    the operators between the matrix products on one [rows, cols] activation: LayerNorm,
             Softmax, ElementBinary add and multiply, Dropout, each forward and backward
  tokens     a token embedding: gather, and the scatter-add of its gradient
  tables     the sparse half of a recommendation model: bags summed from several tables, concatenated
             with the dense features, and the gradients back into the tables
  adam       the Adam update of fp32 master weights with a bf16 copy written out
"""
import ctypes
import importlib
import math

import numpy as np
import torch

ffk = importlib.import_module("flexflow-train_amd")

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
ACTIVATIONS = {"none": ffk.ACT_NONE, "relu": ffk.ACT_RELU, "gelu": ffk.ACT_GELU}


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the reference's CPU-runnable Linear: two calls that are over in microseconds, where the
        # way to the GPU is the cost
        {"name": "linear_small_fp32", "kind": "linear", "dtype": "fp32", "batch": 32, "in": 64, "out": 128,
         "act": "relu"},
        # a language model's vocabulary projection: the widest matrix product of such a model, with
        # as many columns as the vocabulary has entries, which is no round number
        {"name": "linear_vocabulary_bf16", "kind": "linear", "dtype": "bf16", "batch": 2048, "in": 1024,
         "out": 50257, "act": "none"},
        # an encoder layer so small that launches and the gaps between them are what it costs
        {"name": "encoder_small_bf16", "kind": "encoder", "batch": 2, "seq": 48, "d_model": 128, "heads": 2,
         "d_ff": 256, "dropout": 0.1, "pre_ln": True, "act": "gelu", "causal": False, "overwrite": True},
        # the benchmark's training step: one pre-LayerNorm encoder layer at batch 8, 512 tokens
        {"name": "encoder_bf16", "kind": "encoder", "batch": 8, "seq": 512, "d_model": 1024, "heads": 16,
         "d_ff": 4096, "dropout": 0.1, "pre_ln": True, "act": "gelu", "causal": False, "overwrite": True},
        # the reference's order of operators (post-LayerNorm, ReLU, gradients added into) on a batch
        # whose sequence length and token count are odd, as unpadded batches are
        {"name": "encoder_ragged_bf16", "kind": "encoder", "batch": 7, "seq": 197, "d_model": 768, "heads": 12,
         "d_ff": 3072, "dropout": 0.1, "pre_ln": False, "act": "relu", "causal": False, "overwrite": False},
        # attention in the reference's own data type with its model builders' head size of 256
        {"name": "mha_fp32", "kind": "mha", "dtype": "fp32", "batch": 8, "seq": 512, "kv_seq": 512,
         "d_model": 512, "heads": 8, "head_dim": 256, "causal": False},
        # a decoder block's causal attention at full length: the largest matrix work of the set
        {"name": "mha_causal_bf16", "kind": "mha", "dtype": "bf16", "batch": 4, "seq": 4096, "kv_seq": 4096,
         "d_model": 4096, "heads": 32, "head_dim": 128, "causal": True},
        # the bandwidth-bound operators on a large activation
        {"name": "rowwise_bf16", "kind": "rowwise", "dtype": "bf16", "rows": 16384, "cols": 4096},
        # the same on an activation whose rows are neither whole vectors nor whole cache lines
        {"name": "rowwise_ragged_fp32", "kind": "rowwise", "dtype": "fp32", "rows": 3001, "cols": 1001},
        # a language model's token embedding: 65 536 ids of a 50 257-entry vocabulary
        {"name": "tokens_fp32_bf16", "kind": "tokens", "dtype": "bf16", "vocab": 50257, "dim": 1024, "ids": 65536},
        # a recommendation model's tables: eight of a million rows, bags of 32
        {"name": "tables_fp32", "kind": "tables", "tables": 8, "rows": 1000000, "dim": 128, "bags": 16384, "bag": 32},
        # the weights of one encoder layer stepped by Adam from bf16 gradients
        {"name": "adam_bf16", "kind": "adam", "dtype": "bf16", "params": 12596224},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, unit):
    """Spread over the logarithm; half of them multiples of 64, the others any multiple of `unit`."""
    n = _log_uniform(rng, lo, hi)
    unit = 64 if rng.random() < 0.5 and n >= 64 else unit
    return max(unit, n // unit * unit)


def draw(rng):
    kind = rng.choice(("linear", "encoder", "mha", "rowwise", "tokens", "tables", "adam"))
    case = {"kind": kind}
    if kind == "linear":
        case["dtype"] = rng.choice(("bf16", "fp32"))
        case["batch"] = _size(rng, 16, 8192, 1)
        case["in"] = _size(rng, 32, 4096, 1)
        if rng.random() < 0.2:  # a vocabulary
            case["batch"] = min(case["batch"], 2048)
            case["in"] = min(case["in"], 1024)
            case["out"] = rng.randint(5000, 51000)
        else:
            case["out"] = _size(rng, 32, 4096, 1)
        case["batch"] = max(1, min(case["batch"], 100_000_000_000 // (case["in"] * case["out"])))
        case["act"] = rng.choice(("none", "relu"))
    elif kind == "encoder":
        head_dim = rng.choice((32, 64, 64, 64, 80, 128))
        case["heads"] = rng.choice((2, 4, 8, 12, 16))
        case["d_model"] = case["heads"] * head_dim
        case["d_ff"] = rng.choice((2, 4)) * case["d_model"]
        case["batch"] = rng.randint(1, 12)
        case["seq"] = _log_uniform(rng, 16, 700)
        case["dropout"] = rng.choice((0.0, 0.1))
        case["pre_ln"] = rng.random() < 0.5
        case["act"] = rng.choice(("relu", "gelu"))
        case["causal"] = rng.random() < 0.5
        case["overwrite"] = rng.random() < 0.5
    elif kind == "mha":
        case["dtype"] = rng.choice(("bf16", "bf16", "fp32"))
        case["heads"] = rng.choice((4, 8, 16, 32))
        case["head_dim"] = rng.choice((64, 64, 128, 128, 80, 256))
        case["d_model"] = min(4096, case["heads"] * min(case["head_dim"], 128))
        case["batch"] = rng.randint(1, 6)
        case["seq"] = _log_uniform(rng, 32, 2500 if case["dtype"] == "bf16" else 700)
        case["kv_seq"] = case["seq"] if rng.random() < 0.75 else _log_uniform(rng, 32, case["seq"] + 64)
        case["causal"] = case["kv_seq"] == case["seq"] and rng.random() < 0.6
    elif kind == "rowwise":
        case["dtype"] = rng.choice(("bf16", "bf16", "fp32"))
        case["cols"] = _size(rng, 64, 8192, 1)
        case["rows"] = _log_uniform(rng, 64, (1 << 26) // case["cols"] // (1 if case["dtype"] == "bf16" else 2))
    elif kind == "tokens":
        case["dtype"] = rng.choice(("bf16", "fp32"))
        case["vocab"] = _log_uniform(rng, 1000, 120000)
        case["dim"] = _size(rng, 64, 1600, 8)
        case["ids"] = _log_uniform(rng, 200, 65536)
    elif kind == "tables":
        case["tables"] = rng.randint(1, 8)
        case["rows"] = _log_uniform(rng, 10000, 1000000)
        case["dim"] = rng.choice((16, 32, 48, 64, 96, 128))
        case["bags"] = _log_uniform(rng, 200, 16384)
        case["bag"] = _log_uniform(rng, 1, 32)
    else:
        case["dtype"] = rng.choice(("bf16", "fp32"))
        case["params"] = _log_uniform(rng, 20000, 64 << 20)
    return case


# ---------------------------------------------------------------------------
# What a program has in hand before the call
# ---------------------------------------------------------------------------
def _zipf_ids(gen, count, vocab, dtype):
    """Ids drawn Zipf(1.1) over [0, vocab): the frequencies of words and of categorical features."""
    p = torch.arange(1, vocab + 1, device="cuda", dtype=torch.float64) ** -1.1
    cdf = torch.cumsum(p / p.sum(), 0)
    u = torch.rand(count, device="cuda", dtype=torch.float64, generator=gen)
    return torch.searchsorted(cdf, u).clamp_(max=vocab - 1).to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0, dtype=torch.float32):
        t = torch.randn(shape, device="cuda", generator=gen)
        return (t * std if std != 1.0 else t).to(dtype)

    return globals()["_prepare_" + case["kind"]](case, seed, gen, normal)


def _prepare_linear(case, seed, gen, normal):
    dt, B, I, O = DTYPES[case["dtype"]], case["batch"], case["in"], case["out"]
    st = {"act": ACTIVATIONS[case["act"]], "x": normal(B, I, dtype=dt), "w": normal(O, I, std=0.02, dtype=dt),
          "b": normal(O, std=0.02, dtype=dt), "dy": normal(B, O, dtype=dt), "y": torch.empty((B, O), device="cuda", dtype=dt)}
    st["dx"], st["dw"], st["db"] = (torch.empty_like(st[k]) for k in ("x", "w", "b"))
    need = ffk.lib().ffk_linear_backward_workspace_bytes(ffk.dtype_of(st["x"]), st["act"], 1, B, O)
    st["ws"] = torch.empty((max(need, 1),), dtype=torch.uint8, device="cuda")
    st["run"] = _run_linear
    return st


def _prepare_encoder(case, seed, gen, normal):
    bt = torch.bfloat16
    E, H = case["d_model"], case["heads"]
    desc = ffk.EncoderLayerDesc(case["batch"], case["seq"], E, H, case["d_ff"], case["dropout"], seed, 1e-5,
                                1.0 / math.sqrt(E // H), int(case["causal"]), int(case["pre_ln"]),
                                ACTIVATIONS[case["act"]], int(case["overwrite"]))
    w = {}
    for name, shape in ffk.encoder_layer_param_shapes(desc).items():
        t = normal(*shape, std=0.02)
        w[name] = (t + 1.0 if name.endswith("gamma") else t).to(bt)
    g = {name: torch.zeros_like(t) for name, t in w.items()}
    T = case["batch"] * case["seq"]
    x, dy = normal(T, E, dtype=bt), normal(T, E, dtype=bt)
    return {"run": _run_encoder, "desc": desc, "w": w, "g": g, "W": ffk.encoder_layer_params(w),
            "G": ffk.encoder_layer_params(g), "x": x, "dy": dy, "y": torch.empty_like(x), "dx": torch.empty_like(x),
            "ws": ffk.encoder_layer_workspace(desc, ffk.BF16)}


def _prepare_mha(case, seed, gen, normal):
    dt, B, H, D, E = DTYPES[case["dtype"]], case["batch"], case["heads"], case["head_dim"], case["d_model"]
    desc = ffk.mha_desc(B, H, E, E, E, D, D, D, E, case["seq"], case["kv_seq"], 1.0 / math.sqrt(D), case["causal"])
    x = normal(B, case["seq"], E, dtype=dt)
    # self-attention: one tensor in three roles; otherwise the keys and values come from another sequence
    own = case["kv_seq"] == case["seq"]
    kv = x if own else normal(B, case["kv_seq"], E, dtype=dt)
    w = normal(int(ffk.lib().ffk_mha_weight_elements(ctypes.byref(desc))), std=0.02, dtype=dt)
    return {"run": _run_mha, "desc": desc, "x": x, "kv": kv, "w": w, "dout": normal(B, case["seq"], E, dtype=dt),
            "out": torch.empty_like(x), "dx": torch.empty_like(x), "dk": None if own else torch.empty_like(kv),
            "dv": None if own else torch.empty_like(kv), "dw": torch.empty_like(w),
            "reserve": ffk.mha_reserve(desc, ffk.dtype_of(x))}


def _prepare_rowwise(case, seed, gen, normal):
    dt, M, N = DTYPES[case["dtype"]], case["rows"], case["cols"]
    st = {"run": _run_rowwise, "seed": seed, "a": normal(M, N, dtype=dt), "b": normal(M, N, dtype=dt),
          "logits": normal(M, N, std=4.0, dtype=dt), "gamma": (normal(N, std=0.02) + 1.0).to(dt),
          "beta": normal(N, std=0.02, dtype=dt)}
    for name in ("ln", "dln", "p", "dp", "sum", "dadd_l", "dadd_r", "prod", "dmul_l", "dmul_r", "drop", "ddrop"):
        st[name] = torch.empty_like(st["a"])
    st["mean"], st["rstd"] = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    st["dgamma"], st["dbeta"] = torch.empty_like(st["gamma"]), torch.empty_like(st["beta"])
    st["ws"] = torch.empty(ffk.lib().ffk_layer_norm_backward_workspace_bytes(M, N), dtype=torch.uint8, device="cuda")
    return st


def _prepare_tokens(case, seed, gen, normal):
    dt, V, D, n = DTYPES[case["dtype"]], case["vocab"], case["dim"], case["ids"]
    return {"run": _run_tokens, "dtype": dt, "ids": _zipf_ids(gen, n, V, torch.int32), "table": normal(V, D, std=0.02),
            "dy": normal(n, D, dtype=dt), "dtable": torch.zeros((V, D), device="cuda")}


def _prepare_tables(case, seed, gen, normal):
    T, V, D, B, bag = (case[k] for k in ("tables", "rows", "dim", "bags", "bag"))
    return {"run": _run_tables, "tables": [normal(V, D) for _ in range(T)],
            "ids": [_zipf_ids(gen, B * bag, V, torch.int64).view(B, bag) for _ in range(T)],
            "dtables": [torch.zeros((V, D), device="cuda") for _ in range(T)],
            "dense": normal(B, D), "dcat": normal(B, (T + 1) * D), "cat": torch.empty((B, (T + 1) * D), device="cuda"),
            "dparts": [torch.empty((B, D), device="cuda") for _ in range(T + 1)]}


def _prepare_adam(case, seed, gen, normal):
    n = case["params"]
    w = normal(n, std=0.02)
    return {"run": _run_adam, "w": w, "grad": normal(n, std=1e-3, dtype=DTYPES[case["dtype"]]),
            "m": torch.zeros(n, device="cuda"), "v": torch.zeros(n, device="cuda"), "w_bf16": w.to(torch.bfloat16)}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    return state["run"](state)


def _run_linear(s):
    ffk.linear_forward(s["x"], s["w"], s["b"], s["act"], out=s["y"])
    ffk.linear_backward(s["y"], s["dy"], s["x"], s["w"], s["dx"], s["dw"], s["db"], activation=s["act"], workspace=s["ws"])
    return s["y"], s["dx"], s["dw"], s["db"]


def _run_encoder(s):
    ffk.encoder_layer_forward(s["desc"], s["W"], s["x"], s["y"], s["ws"])
    ffk.encoder_layer_backward(s["desc"], s["W"], s["G"], s["x"], s["dy"], s["dx"], s["ws"])
    return s["y"], s["dx"], s["g"]


def _run_mha(s):
    x, kv = s["x"], s["kv"]
    ffk.mha_forward(s["desc"], x, kv, kv, s["w"], s["reserve"], out=s["out"])
    ffk.mha_backward(s["desc"], x, s["dx"], kv, s["dk"], kv, s["dv"], s["w"], s["dw"], s["dout"], s["reserve"],
                     accumulate=ffk.MHA_OVERWRITE_WEIGHT_GRAD)
    return s["out"], s["dx"], s["dk"], s["dv"], s["dw"]


def _run_rowwise(s):
    a, b, rows, cols = s["a"], s["b"], s["a"].shape[0], s["a"].shape[1]
    ffk.layer_norm_forward(a, s["gamma"], s["beta"], 1e-5, s["ln"], s["mean"], s["rstd"])
    ffk.layer_norm_backward(b, a, s["mean"], s["rstd"], s["gamma"], s["dln"], s["dgamma"], s["dbeta"], workspace=s["ws"])
    ffk.softmax_forward(s["logits"], rows, cols, 1, out=s["p"])
    ffk.softmax_backward(s["p"], b, rows, cols, 1, dx=s["dp"])
    ffk.element_binary_forward(ffk.OP["EW_ADD"], a, b, out=s["sum"])
    ffk.element_binary_backward(ffk.OP["EW_ADD"], s["logits"], a, b, s["dadd_l"], s["dadd_r"])
    ffk.element_binary_forward(ffk.OP["EW_MUL"], a, b, out=s["prod"])
    ffk.element_binary_backward(ffk.OP["EW_MUL"], s["logits"], a, b, s["dmul_l"], s["dmul_r"])
    ffk.dropout_forward(a, 0.1, s["seed"], out=s["drop"])
    ffk.dropout_backward(b, 0.1, s["seed"], dx=s["ddrop"])
    return [s[k] for k in ("ln", "mean", "rstd", "dln", "dgamma", "dbeta", "p", "dp", "sum", "dadd_l", "dadd_r",
                           "prod", "dmul_l", "dmul_r", "drop", "ddrop")]


def _run_tokens(s):
    out = ffk.embedding_forward(s["ids"], s["table"], out_dtype=s["dtype"])
    ffk.embedding_backward(s["ids"], s["dy"], s["dtable"])
    return out, s["dtable"]


def _run_tables(s):
    pooled = [ffk.embedding_forward(i, t, aggr=ffk.AGGR_SUM) for i, t in zip(s["ids"], s["tables"])]
    ffk.concat_forward(pooled + [s["dense"]], 1, out=s["cat"])
    ffk.concat_backward(s["dcat"], s["dparts"], 1, accumulate=False)
    for i, dy, dt in zip(s["ids"], s["dparts"], s["dtables"]):
        ffk.embedding_backward(i, dy, dt, aggr=ffk.AGGR_SUM)
    return s["cat"], s["dparts"][-1], s["dtables"]


def _run_adam(s):
    ffk.adam_update(s["w"], s["grad"], s["m"], s["v"], 1e-4, weight_decay=1e-2, weight_lowp=s["w_bf16"])
    return s["w"], s["m"], s["v"], s["w_bf16"]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far correct results may lie apart
# ---------------------------------------------------------------------------
def _touched(count, vocab):
    """Expected number of different ids among `count` draws of _zipf_ids."""
    p = np.arange(1, vocab + 1, dtype=np.float64) ** -1.1
    p /= p.sum()
    return float(np.sum(-np.expm1(count * np.log1p(-p))))


def work(case):
    kind = case["kind"]
    es = {"bf16": 2, "fp32": 4}[case.get("dtype", "bf16")]
    if kind == "linear":
        B, I, O = case["batch"], case["in"], case["out"]
        return {"bytes": es * (2 * B * I + 2 * O * I + 2 * B * O + 2 * O), "flops": 6.0 * B * I * O}
    if kind == "encoder":
        T, E, F = case["batch"] * case["seq"], case["d_model"], case["d_ff"]
        core = 4.0 * T * case["seq"] * E * (0.5 if case["causal"] else 1.0)
        params = 4 * E * E + 2 * E * F + 5 * E + F
        grads = 1 if case["overwrite"] else 2
        return {"bytes": 2.0 * (4 * T * E + (1 + grads) * params), "flops": 3.0 * (2.0 * T * (4 * E * E + 2 * E * F) + core)}
    if kind == "mha":
        B, Sq, Sk, E, HD = case["batch"], case["seq"], case["kv_seq"], case["d_model"], case["heads"] * case["head_dim"]
        core = 4.0 * B * Sq * Sk * HD * (0.5 if case["causal"] else 1.0)
        own = Sq == Sk
        return {"bytes": float(es) * (4 * B * Sq * E + (0 if own else 3 * B * Sk * E) + 2 * 4 * HD * E),
                "flops": 3.0 * (2.0 * B * (2 * Sq + 2 * Sk) * E * HD + core)}
    if kind == "rowwise":
        # LayerNorm 2 + 3 tensors, Softmax 2 + 3, add 3 + 3, multiply 3 + 5, Dropout 2 + 2
        return {"bytes": 28.0 * es * case["rows"] * case["cols"], "flops": 0}
    if kind == "tokens":
        n, D, rows = case["ids"], case["dim"], _touched(case["ids"], case["vocab"])
        return {"bytes": 4.0 * n + 4.0 * rows * D + es * n * D + 4.0 * n + es * n * D + 8.0 * rows * D, "flops": 0}
    if kind == "tables":
        T, D, B = case["tables"], case["dim"], case["bags"]
        n, rows = B * case["bag"], _touched(B * case["bag"], case["rows"])
        concat = 4.0 * B * D * (T + 1)
        return {"bytes": T * (16.0 * n + 12.0 * rows * D) + 3 * concat, "flops": 0}
    return {"bytes": case["params"] * (24.0 + es + 2.0), "flops": 0}


def tolerance(case):
    if case["kind"] in ("linear", "encoder", "mha", "rowwise") and case.get("dtype", "bf16") == "bf16":
        return {"rel": 1e-2}
    if case["kind"] == "tokens" and case["dtype"] == "bf16":
        return {"rel": 4e-3}  # a gather rounded to bf16, and fp32 sums
    return {"rel": 1e-5}
