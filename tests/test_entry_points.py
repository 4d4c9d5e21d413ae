"""What the entry points do with arguments that are no dense tensors of the device: a Python error,
before anything is launched.  Fake tensors stand in for the device's, so no GPU is needed."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import sys
sys.path[:0] = [%r]
import importlib
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
ffk = importlib.import_module("flexflow-train_amd")

def refused(what, kind, call):
    try:
        call()
    except kind as e:
        print("refused", what, type(e).__name__, flush=True)
    else:
        raise SystemExit(what + " was accepted")
""" % ROOT


def run(body):
    """In a process of its own: a C++ exception that leaves an entry point would end it."""
    done = subprocess.run([sys.executable, "-c", PRELUDE + body], capture_output=True, text=True, timeout=300,
                          cwd=ROOT)
    assert done.returncode == 0, (done.returncode, done.stdout[-1000:], done.stderr[-1000:])
    return done.stdout


@pytest.mark.parametrize("call", [
    "ffk.softmax_forward(t, 1, 8, 1)",
    "ffk.dropout_forward(t, 0.1, 1)",
    "ffk.layer_norm_forward(t.view(1, 8), None, None, 1e-5)",
])
def test_tensor_without_an_address(call):
    """torch.vmap's tensors have none: torch's exception arrives as a RuntimeError."""
    out = run("""
with FakeTensorMode():
    x = torch.empty((4, 8), device="cuda")
    refused("vmap", RuntimeError, lambda: torch.vmap(lambda t: %s)(x))
""" % call)
    assert out.strip() == "refused vmap RuntimeError"
