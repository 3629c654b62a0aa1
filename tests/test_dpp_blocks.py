"""CPU: the row broadcasts of the factor's diagonal blocks keep their wait states.

A DPP operand needs two wait states after a VALU instruction writes its
register, and the compiler inserts none inside inline assembly.  The listing of
the diagonal block's code (compiled here, not run) must have every such
statement spend two states before its first broadcast, and no DPP instruction
anywhere within two wait states of a VALU write of its operand.
"""
import os
import re
import subprocess

import pytest

from g2ptq_amd import build

SOURCE = """
#include "common.hpp"
#include "potrf.hpp"
using namespace g2ptq;
extern "C" __global__ __launch_bounds__(256) void diag_block(const float* in, float* out, int* f) {
  __shared__ float Xs[POT_NB * XP];
  __shared__ __attribute__((aligned(16))) float Lm[POT_NB * LP];
  __shared__ __attribute__((aligned(16))) float rdv[POT_NB];
  __shared__ int fs;
  for (int e = threadIdx.x; e < POT_NB * XP; e += 256) Xs[e] = in[e];
  __syncthreads();
  *f = potrf_core(Xs, Lm, rdv, &fs);
  for (int e = threadIdx.x; e < POT_NB * XP; e += 256) out[e] = Xs[e];
}
"""


def _listing(tmp_path):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    src, out = tmp_path / "diag.hip", tmp_path / "diag.s"
    src.write_text(SOURCE)
    subprocess.run([build.HIPCC, *build.FLAGS, "-I", build.CSRC, "--offload-device-only", "-S",
                    str(src), "-o", str(out)], check=True, capture_output=True, timeout=300)
    return out.read_text()


def _instructions(text):
    """(opcode, operands, number of its inline statement or None) in order; inline
    `.if` blocks that the assembler leaves out are left out here."""
    found, block, inline, keep = [], 0, False, True
    body = text[text.index("diag_block:"):text.index(".Lfunc_end0")]
    for line in body.splitlines():
        line = line.strip()
        if "#ASMSTART" in line:
            block, inline, keep = block + 1, True, True
        elif "#ASMEND" in line:
            assert keep
            inline = False
        elif m := re.match(r"\.if (\d+) (>=|>|==) (\d+)$", line):
            a, b = int(m[1]), int(m[3])
            keep = {">=": a >= b, ">": a > b, "==": a == b}[m[2]]
        elif line == ".endif":
            keep = True
        elif keep and re.match(r"[a-z]+_\w+", line):
            code = line.split(";")[0].split(None, 1)
            found.append((code[0], code[1] if len(code) > 1 else "", block if inline else None))
    return found


def _registers(operand):
    """The vector registers of an operand such as -v7 or v[8:11]."""
    if m := re.match(r"-?\|?v\[(\d+):(\d+)\]", operand):
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"-?\|?v(\d+)", operand)
    return {int(m[1])} if m else set()


def _operands(args):
    return [a.strip().split(" ")[0] for a in args.split(",")]


def test_row_broadcasts_wait_for_their_operand(tmp_path):
    code = _instructions(_listing(tmp_path))
    dpp = 0
    recent = []  # (wait states since, registers) of the VALU writes that still count
    statement, inside = None, 0  # the inline statement, and the states spent in it
    for op, args, block in code:
        if block != statement:
            statement, inside = block, 0
        ops = _operands(args)
        if "_dpp" in op:
            dpp += 1
            source = _registers(ops[1])
            assert not any(source & regs for _, regs in recent), (op, args, "too soon")
            assert block is None or inside >= 2, \
                (op, args, "an inline statement has to wait before its first broadcast")
        states = int(args) + 1 if op == "s_nop" else 1
        inside += states
        recent = [(n + states, r) for n, r in recent if n + states < 2]
        if op.startswith("v_") and not op.startswith(("v_cmp", "v_mfma", "v_readlane",
                                                      "v_readfirstlane")):
            recent.append((0, _registers(ops[0])))
    # per panel 2·(15 + … + 1) updates and 16 pivots, and the inverse's chains
    assert dpp > 240
