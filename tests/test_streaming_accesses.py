"""Kernels that are meant to read or write past the caches do so in the built library: the hint is lost
without a word where the compiler finds an access without it at the same address."""
import glob
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin/"
# kernel -> which of its boolean template arguments asks for it, whether its stores are meant too
KERNELS = {"softmax_fwd_kernel": (0, True), "softmax_bwd_kernel": (0, True),
           "layer_norm_fwd_kernel": (1, True), "layer_norm_bwd_kernel": (3, False)}
NAME = re.compile(r"\d(%s)I(?:f|DF16b)Li\d+ELi\d+E((?:Lb[01]E)+)E" % "|".join(KERNELS))


def out(*cmd, **kw):
    return subprocess.run(cmd, capture_output=True, text=True, check=True, **kw).stdout


@pytest.mark.skipif(not os.path.exists(LLVM + "llvm-objdump"), reason="no disassembler here")
def test_row_kernels_stream(ffk, tmp_path):
    shutil.copy(ffk.LIB_PATH, tmp_path / "lib.so")
    out(LLVM + "llvm-objdump", "--offloading", "lib.so", cwd=tmp_path)
    seen = set()
    for path in glob.glob(str(tmp_path / "lib.so.*gfx950")):
        names = [n for n in re.findall(r" T (\S+)$", out("nm", path), re.M) if NAME.search(n)]
        if not names:
            continue
        text = out(LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names), path)
        for name, body in re.findall(r"<(\S+)>:\n(.*?)(?=\n\n|\Z)", text, re.S):
            kernel, flags = NAME.search(name).groups()
            which, stores = KERNELS[kernel]
            stream = flags[4 * which + 2] == "1"
            loads = len(re.findall(r"global_load_dwordx4 .*\bnt\b", body))
            written = len(re.findall(r"global_store_dwordx4 .*\bnt\b", body))
            assert (loads > 0) == stream and (written > 0) == (stream and stores), (name, loads, written)
            seen.add((kernel, stream))
    assert seen == {(k, s) for k in KERNELS for s in (False, True)}


@pytest.mark.skipif(not os.path.exists(LLVM + "llvm-objdump"), reason="no disassembler here")
def test_embedding_gradients_read_once_stream(ffk, tmp_path):
    """The walk over sorted lookups reads a gradient row past the caches where each stands for one lookup, and where
    bags read theirs again, through them."""
    shutil.copy(ffk.LIB_PATH, tmp_path / "lib.so")
    out(LLVM + "llvm-objdump", "--offloading", "lib.so", cwd=tmp_path)
    pattern = re.compile(r"embedding_bwd_walk_kernelIDF16bLi(\d+)ELb([01])E")  # its 8-byte loads are the gradient's
    seen = set()
    for path in glob.glob(str(tmp_path / "lib.so.*gfx950")):
        names = [n for n in re.findall(r" T (\S+)$", out("nm", path), re.M) if pattern.search(n)]
        if not names:
            continue
        text = out(LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(names), path)
        for name, body in re.findall(r"<(\S+)>:\n(.*?)(?=\n\n|\Z)", text, re.S):
            lanes, bagged = pattern.search(name).groups()
            rows = re.findall(r"buffer_load_dwordx2 .*", body)
            past = [r for r in rows if re.search(r"\bnt\b", r)]
            assert rows and past == (rows if bagged == "0" else []), (name, rows)
            seen.add((int(lanes), bagged))
    assert seen == {(lanes, b) for lanes in (4, 8, 16, 32, 64) for b in "01"}
