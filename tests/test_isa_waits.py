"""The wait states of the inline-assembly MFMAs (gemm.hip, mfma_group) in the code as built: the
compiler inserts none for instructions that it does not see. Read from the disassembly of this tree's
own library; no GPU."""
import os
import re
import shutil
import subprocess

import pytest

from deepgemm_amd import build

MFMA = "v_mfma_f32_16x16x128_f8f6f4"
# wait states from an MFMA to a read of its result: 11 after 8 passes (this one), 19 after 16
RESULT_WAIT = 19
OPERAND_WAIT = 2  # from a VALU write of an operand to the MFMA


def _objdump():
    found = [os.path.join(os.path.dirname(os.path.realpath(build._hipcc())), "..", *p, "llvm-objdump")
             for p in (("llvm", "bin"), ("lib", "llvm", "bin"))]
    tool = next((p for p in found if os.path.exists(p)), shutil.which("llvm-objdump"))
    if tool is None:
        pytest.skip("llvm-objdump is not installed")
    return tool


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: [(address, opcode, operands, branch target or None)]} of the kernels with that MFMA."""
    if not os.path.exists(build.LIB_PATH):
        build.build()
    where = tmp_path_factory.mktemp("isa")
    lib = shutil.copy(build.LIB_PATH, where)
    subprocess.run([_objdump(), "--offloading", lib], check=True, capture_output=True, cwd=where)
    out = {}
    for name in sorted(os.listdir(where)):
        if not name.endswith(build.ARCH):
            continue
        text = subprocess.run([_objdump(), "-d", "--no-show-raw-insn", str(where / name)], check=True,
                              capture_output=True, text=True).stdout
        for body in re.split(r"\n\n(?=[0-9a-f]{16} <)", text):
            if MFMA not in body:
                continue
            head = re.search(r"([0-9a-f]{16}) <(\S+)>:", body)
            base, code = int(head[1], 16), []
            for line in body.splitlines():
                m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):.*?(?:<\S+?\+0x([0-9a-f]+)>)?$", line)
                if m:
                    code.append((int(m[3], 16), m[1], m[2], base + int(m[4], 16) if m[4] else None))
            out[head[2]] = code
    assert out, "no kernel with inline-assembly MFMAs found"
    return out


def _states(op, args):
    return int(args, 0) + 1 if op == "s_nop" else 1


def _regs(args):
    """The vector and accumulation registers named in a list of operands: {"v34", "a0", ...}."""
    regs = set()
    for kind, lo, hi, one in re.findall(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)", args):
        regs.update(f"{kind}{r}" for r in (range(int(lo), int(hi) + 1) if lo else (int(one),)))
    return regs


def _written(op, args):
    """The vector registers that a VALU instruction writes, as names."""
    if not op.startswith("v_") or op.startswith(("v_mfma", "v_cmp", "v_readfirstlane", "v_readlane")):
        return set()
    return _regs(",".join(args.split(",")[:2 if op.startswith("v_swap") else 1]))


def test_operands_are_not_written_right_before(kernels):
    """A VALU write of an operand needs OPERAND_WAIT wait states before the MFMA, along every path
    that leads to it."""
    for name, code in kernels.items():
        before = {i: [i - 1] for i in range(1, len(code)) if code[i - 1][1] not in ("s_branch", "s_endpgm")}
        at = {addr: i for i, (addr, *_) in enumerate(code)}
        for i, (_, op, args, target) in enumerate(code):
            if op.startswith(("s_branch", "s_cbranch")):
                before.setdefault(at[target], []).append(i)
        for i, (_, op, args, _) in enumerate(code):
            if op != MFMA:
                continue
            operands, todo = _regs(args), [(j, 0) for j in before.get(i, [])]
            while todo:
                j, states = todo.pop()
                _, jop, jargs, _ = code[j]
                assert not (operands & _written(jop, jargs)), f"{name}: {jop} {jargs}, {states} wait states, {args}"
                states += _states(jop, jargs)
                if states < OPERAND_WAIT:
                    todo += [(k, states) for k in before.get(j, [])]


def test_no_accumulator_is_touched_before_its_result(kernels):
    """From every MFMA along every path, for as many wait states as a result may take: no other
    instruction reads or writes its accumulators."""
    for name, code in kernels.items():
        at = {addr: i for i, (addr, *_) in enumerate(code)}
        for i, (_, op, args, _) in enumerate(code):
            if op != MFMA:
                continue
            acc = _regs(args.split(",")[0])
            assert len(acc) == 4 and all(r[0] == "a" for r in acc), f"{name}: {args}"
            todo, seen = [(i + 1, 0)], set()
            while todo:
                j, states = todo.pop()
                if states >= RESULT_WAIT or j >= len(code) or (j, states) in seen:
                    continue
                seen.add((j, states))
                _, jop, jargs, target = code[j]
                if jop != MFMA:
                    assert not (acc & _regs(jargs)), f"{name}: {jop} {jargs} {states} wait states after {args}"
                states += _states(jop, jargs)
                if jop.startswith(("s_branch", "s_cbranch")):
                    assert target in at, f"{name}: {jop} {jargs}"
                    todo.append((at[target], states))
                if jop not in ("s_branch", "s_endpgm"):
                    todo.append((j + 1, states))
