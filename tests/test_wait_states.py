"""Instructions written out in the kernels' sources keep the distances that the hardware asks for, in the built library: the
compiler neither sees what they do nor puts wait states in front of them.

  * direct loads (csrc/lds_dma.h): five wait states between a vector instruction that writes a scalar register and a
    vector-memory instruction that reads it; one between a write of M0 and the direct load behind it
  * matrix instructions with the accumulator in place (csrc/gemm_bf16.h): see the second test
"""
import functools
import glob
import os
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin/"
pytestmark = pytest.mark.skipif(not os.path.exists(LLVM + "llvm-objdump"), reason="no disassembler here")

KERNEL = re.compile(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^\n|\Z)", re.S | re.M)
LINE = re.compile(r"^\t(\S+)([^/\n]*?)\s*// ([0-9A-F]+):.*?(?:<\S+\+0x([0-9a-f]+)>)?$", re.M)
REGISTER = re.compile(r"\b([sva])(?:(\d+)\b|\[(\d+):(\d+)\])|\b(vcc|m0)\b")
# vector instructions with a scalar destination behind the vector one (carries, scales)
SECOND = re.compile(r"v_(add|sub|subrev|addc|subb|subbrev)_co|v_div_scale|v_mad_[ui]64_[ui]32")


@functools.lru_cache(maxsize=None)
def registers(operand):
    out = set()
    for kind, one, first, last, name in REGISTER.findall(operand):
        if name:
            out.add(name)
        else:
            out.update((kind, i) for i in range(int(one or first), int(one or last) + 1))
    return out


class Code:
    """The instructions of one kernel, and which can come before which."""

    def __init__(self, text):
        lines = LINE.findall(text)
        self.op = [op for op, _, _, _ in lines]
        self.args = [[a.strip() for a in re.split(r",(?![^\[]*\])", args)] if args.strip() else [] for _, args, _, _ in lines]
        address = [int(a, 16) for _, _, a, _ in lines]
        at = {a: i for i, a in enumerate(address)}
        self.before = [[] for _ in lines]
        for i, (op, _, _, target) in enumerate(lines):
            if op.startswith(("s_cbranch", "s_branch")):
                self.before[at[address[0] + int(target or "0", 16)]].append(i)
            if i + 1 < len(lines) and not op.startswith(("s_branch", "s_endpgm", "s_setpc")):
                self.before[i + 1].append(i)

    def wait_states(self, i):
        return int(self.args[i][0], 0) + 1 if self.op[i] == "s_nop" else 1

    def scalar_writes(self, i):
        """(scalar registers that instruction i writes, whether it is a vector instruction)"""
        op, args = self.op[i], self.args[i]
        if op.startswith("v_"):
            out = registers(args[0]) if args else set()
            if SECOND.match(op):
                out = out | registers(args[1])
            return {r for r in out if r in ("vcc", "m0") or r[0] == "s"}, True
        if op.startswith("s_") and args and not op.startswith(("s_cmp", "s_bitcmp", "s_waitcnt", "s_nop", "s_cbranch", "s_branch")):
            return registers(args[0]), False
        return set(), False

    def vector_written(self, i, wanted, states):
        """Instructions that reach i with a vector write of one of `wanted` fewer than `states` wait states before it."""
        found, work, seen = [], [(p, wanted, 0) for p in self.before[i]], set()
        while work:
            at, regs, passed = work.pop()
            if (at, frozenset(regs), passed) in seen or passed >= states:
                continue
            seen.add((at, frozenset(regs), passed))
            written, vector = self.scalar_writes(at)
            if vector and written & regs:
                found.append((at, passed))
            left = regs - written
            if left:
                work += [(p, left, passed + self.wait_states(at)) for p in self.before[at]]
        return found


def disassembled(lib, where):
    """(name, instructions) of the library's kernels that have direct loads."""
    shutil.copy(lib, where / "lib.so")
    subprocess.run([LLVM + "llvm-objdump", "--offloading", "lib.so"], cwd=where, check=True, capture_output=True)
    for path in sorted(glob.glob(str(where / "lib.so.*gfx950"))):
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", path], check=True, capture_output=True, text=True).stdout
        for name, body in KERNEL.findall(text):
            if " lds" in body:
                yield name, Code(body)


@pytest.fixture(scope="module")
def kernels(ffk, tmp_path_factory):
    return list(disassembled(ffk.LIB_PATH, tmp_path_factory.mktemp("library")))


def test_direct_loads_read_settled_scalars(kernels):
    checked, wrong = 0, {}
    for name, code in kernels:
        for i, op in enumerate(code.op):
            if not op.startswith("buffer_load") or not code.args[i][-1].endswith("lds"):
                continue
            checked += 1
            scalars = registers(code.args[i][1]) | registers(code.args[i][2])
            for at, passed in code.vector_written(i, {r for r in scalars if r[0] == "s"}, 5):
                wrong.setdefault(name, []).append((code.op[at], code.args[at], passed, code.args[i]))
            # M0 is written by scalar moves; none right in front
            assert not (code.op[i - 1].startswith("s_mov") and code.args[i - 1][0] == "m0"), (name, i)
    assert checked > 1000
    assert not wrong, "%d of %d loads, in %d kernels, for instance %s" % (
        sum(map(len, wrong.values())), checked, len(wrong), [(k, v[0]) for k, v in wrong.items()][:4])


def test_accumulators_written_out_are_settled(kernels):
    """csrc/gemm_bf16.h's matrix instructions with the accumulator in place (v_mfma_f32_16x16x32_bf16, four passes): eight wait
    states before anything but another of them touches a result, two behind a vector instruction that writes an operand.
    Twice as many are asked for here, and kept."""
    op_name, settles, operands = "v_mfma_f32_16x16x32_bf16", 16, 4
    checked, wrong = 0, []
    for name, code in kernels:
        if not any(op == op_name and args[0].startswith("a[") for op, args in zip(code.op, code.args)):
            continue
        used = [frozenset().union(*map(registers, args)) for args in code.args]
        results = {i: registers(code.args[i][0]) for i, op in enumerate(code.op) if op == op_name}
        touches = frozenset().union(*results.values())
        for i, op in enumerate(code.op):
            matrix = op == op_name
            if matrix:
                # what its operands or its accumulator were written by
                wanted, states = frozenset().union(*(registers(a) for a in code.args[i][1:4])), operands
            elif not op.startswith("s_") and used[i] & touches:
                wanted, states = used[i] & touches, settles
            else:
                continue
            checked += 1
            work, seen = [(p, 0) for p in code.before[i]], set()
            while work:
                at, passed = work.pop()
                if (at, passed) in seen or passed >= states:
                    continue
                seen.add((at, passed))
                if matrix:
                    bad = code.op[at].startswith("v_") and not code.op[at].startswith("v_mfma") and registers(code.args[at][0]) & wanted
                else:
                    bad = at in results and results[at] & wanted
                if bad:
                    wrong.append((name, code.op[at], code.args[at], op, code.args[i], passed))
                work += [(p, passed + code.wait_states(at)) for p in code.before[at]]
    assert checked > 10000
    assert not wrong, "%d of %d, for instance %s" % (len(wrong), checked, wrong[:3])
