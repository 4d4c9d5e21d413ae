"""The C-ABI library loads and exports every symbol include/ffk.h declares
(no compute calls: runs without a GPU)."""
import ctypes
import os
import random
import re
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "ffk.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ffk_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_symbol_is_exported(ffk):
    names = _declared_symbols()
    assert len(names) > 30
    handle = ctypes.CDLL(ffk.LIB_PATH)
    missing = [n for n in names if not hasattr(handle, n)]
    assert not missing, missing


def test_python_signature_table_matches_header(ffk):
    assert sorted(ffk.SIGNATURES) == _declared_symbols()


def test_argument_checks_do_not_need_a_device(ffk):
    lib = ffk.lib()
    # preconditions are checked before any HIP call is made
    assert lib.ffk_linear_forward(None, ffk.FLOAT, 7, None, None, None, None, 1, 1, 1) == 1
    assert b"Unhandled activation" in lib.ffk_last_error()
    assert lib.ffk_dropout_forward(None, ffk.FLOAT, None, None, 10, 1.5, 0, 0) == 1
    assert lib.ffk_embedding_forward(None, ffk.INT32, ffk.FLOAT, ffk.FLOAT, None, None, None,
                                     ffk.AGGR_NONE, 4, 2, 8, 10) == 1
    assert lib.ffk_element_unary_forward(None, ffk.FLOAT, 9999, 0.0, 1, 1, 4) == 3
    assert lib.ffk_gemm(None, ffk.DOUBLE, 0, 0, 4, 4, 4, 1, 1, 1, 0) == 3


@pytest.mark.skipif(torch.cuda.is_available(), reason="the addresses are made up")
@pytest.mark.parametrize("shape", [(64, 128, 40), (33, 72, 40), (57, 56, 64), (65, 63, 129), (300, 127, 200)])
def test_linear_backward_refuses_a_call_without_its_scratch(ffk, shape):
    """bf16: an activation's gradient and the bias gradient's partial sums need scratch at every size and alignment,
    whichever kernels run."""
    batch, in_dim, out_dim = shape
    y, dy, x, dx, w, dw, db, ws = (ctypes.c_void_p((i + 1) << 24) for i in range(8))

    def call(act, bias, room):
        return ffk.lib().ffk_linear_backward(None, ffk.BF16, act, 0, y, dy, x, dx, w, dw, db if bias else None, batch,
                                             in_dim, out_dim, ws if room else None, room, 0)

    for act, bias in ((ffk.ACT_RELU, True), (ffk.ACT_RELU, False), (ffk.ACT_NONE, True)):
        for room in (0, 64):
            assert call(act, bias, room) == 4, (act, bias, room)
            assert b"workspace" in ffk.lib().ffk_last_error()


def test_linear_backward_asks_for_split_scratch_it_can_use(ffk):
    """bf16: reductions of up to 18 k-tiles of 64 stay whole, and an encoder layer's Linear backwards are sequences of
    products, whose reductions of up to 63 tiles do.  Neither has a use for the 8 MB of partial sums."""
    lib = ffk.lib()

    def linear(batch, out_dim):
        return lib.ffk_linear_backward_workspace_bytes(ffk.BF16, ffk.ACT_NONE, 0, batch, out_dim)

    assert linear(1152, 1152) == 0
    assert linear(1153, 64) == linear(64, 1160) == 8 << 20

    def layer(tokens):
        desc = ffk.EncoderLayerDesc(1, tokens, 256, 4, 1024)
        return lib.ffk_encoder_layer_workspace_bytes(ctypes.byref(desc), ffk.BF16)

    for tokens in (512, 1153):
        assert 0 < layer(tokens) - layer(tokens - 1) < 1 << 20, tokens


def test_gemm_kernel_name_needs_no_device(ffk):
    """The dispatch answers which kernel a shape runs on without launching anything."""
    big = ffk.gemm_kernel_name(ffk.BF16, False, True, 4096, 4096, 1024, has_bias=True)
    assert big.startswith("gemm_bf16_pipe_kernel<256,256,") and big.endswith("false,true,0,false>")
    assert ffk.gemm_kernel_name(ffk.BF16, True, False, 1024, 1024, 4096).startswith("gemm_bf16_pipe_kernel<128,128,")
    assert ffk.gemm_kernel_name(ffk.FLOAT, False, True, 32, 128, 64, has_bias=True).startswith("gemm_f32_kernel")
    assert ffk.gemm_kernel_name(ffk.BF16, False, False, 51, 131, 251) == "gemm_bf16_plain_kernel"
    # an activation changes the instance, and the answer follows the option that forces a tile
    relu = ffk.gemm_kernel_name(ffk.BF16, False, True, 4096, 4096, 1024, True, ffk.ACT_RELU)
    assert relu != big
    ffk.set_option(ffk.OPTION_GEMM_VARIANT, 128)
    try:
        assert ffk.gemm_kernel_name(ffk.BF16, False, True, 4096, 4096, 1024, True).startswith("gemm_bf16_pipe_kernel<128,128,")
    finally:
        ffk.set_option(ffk.OPTION_GEMM_VARIANT, 0)


def _kernels(path):
    """The kernels in the library: name -> the template argument lists it is instantiated with."""
    symbols = subprocess.run(["nm", "-C", path], capture_output=True, text=True, check=True).stdout
    found = {}
    for name, args in re.findall(r" V (?:void )?ffk::(gemm_\w+_kernel)(?:<([^>]*)>)?\(", symbols):
        found.setdefault(name, set()).add(tuple(args.replace(" ", "").split(",")))
    # what the demangler does not know (_Float16's kin): its literals by hand
    for name, args in re.findall(r" V _ZN3ffk\d+(gemm_\w+_kernel)I((?:L[bi]\d+E)+)E", symbols):
        literals = re.findall(r"L([bi])(\d+)E", args)
        found.setdefault(name, set()).add(tuple(v if t == "i" else ("false", "true")[int(v)] for t, v in literals))
    return found


def test_gemm_kernel_names_are_kernels_of_the_library(ffk):
    """Every name is an instance in the library, arguments left out at the end having their default."""
    have = _kernels(ffk.LIB_PATH)
    defaults = {"gemm_bf16_pipe_kernel": ("0", "1"), "gemm_bf16_plain_kernel": ("64",)}
    rng, seen, launches = random.Random(0), set(), set()
    sizes = [1, 8, 63, 64, 128, 200, 256, 500, 768, 1024, 1379, 2048, 4096, 5000, 8457]
    shapes = [tuple(rng.choice(sizes) for _ in range(3)) for _ in range(400)] + [(2048, 8457, 1024), (4096, 3072, 1024), (51, 131, 9)]
    for dtype in (ffk.FLOAT, ffk.BF16):
        for M, N, K in shapes:
            for ta, tb in ((False, False), (False, True), (True, False), (True, True)):
                names = ffk.gemm_kernel_name(dtype, ta, tb, M, N, K).split(" + ")
                launches.add(len(names))
                for full in names:
                    name, _, args = full.rstrip(">").partition("<")
                    args = tuple(args.split(",")) if args else ()
                    kernel = have.get(name)
                    assert kernel, full
                    n = len(next(iter(kernel)))
                    fill = defaults.get(name, ())
                    args += fill[len(fill) - (n - len(args)):] if n > len(args) else ()
                    assert args in kernel, (full, args)
                    seen.add(name)
    assert launches == {1, 2}
    assert seen == {"gemm_bf16_pipe_kernel", "gemm_bf16_kernel", "gemm_bf16_plain_kernel", "gemm_f32_kernel",
                    "gemm_f32_tiled_kernel", "gemm_f32_small_kernel", "gemm_f32_deep_kernel"}
