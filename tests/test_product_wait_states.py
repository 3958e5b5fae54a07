"""Matrix products written as assembly statements: the wait states around them, which the compiler does not see, in the built code.

An 8-pass product (16x16x32 in bfloat16) reads an operand that an ordinary vector instruction wrote no sooner than two states
before, and its result is read or overwritten by anything but a product no sooner than eleven states behind it. The kernels keep
these by statements of their own; a compiler that put a copy between two of them would break that without a word."""
import os
import re
import subprocess

import pytest

from reinfer_amd.csrc import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
BEFORE, BEHIND = 2, 11


def registers(operand):
    m = re.match(r"[-|]*([va])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return set()
    first = int(m.group(2) or m.group(3))
    return {(m.group(1), i) for i in range(first, int(m.group(2) or m.group(4)) + 1)}


def functions(text):
    """{name: ([(operation, operands)], {label: index})}"""
    out = {}
    for line in text.splitlines():
        line = line.split("//")[0].strip()
        if m := re.fullmatch(r"(?:[0-9a-f]+ )?<([^>]+)>:", line):
            if re.fullmatch(r"L\d+", m.group(1)):
                out[name][1][m.group(1)] = len(out[name][0])
            else:
                name = m.group(1)
                out[name] = ([], {})
        elif out and line and not line.startswith(("Disassembly", ";")):
            op, _, rest = line.partition(" ")
            out[name][0].append((op, [o.strip() for o in rest.split(",")]))
    return out


def breaches(code, labels):
    """(index, index) of instructions that follow one another too closely, along every path. A branch on a scalar pair that the path
    has just set to 0 or -1 (how the compiler leaves a loop that may not have run) goes one way."""
    found = []

    def product(op):
        return op.startswith(("v_mfma", "v_smfma"))

    def walk(start, most, visit):
        todo = [(start + 1, 0, {})]
        while todo:
            i, states, known = todo.pop()
            while i < len(code) and states < most:
                op, args = code[i]
                if visit(op, args):
                    found.append((start, i))
                    break
                if op == "s_mov_b64":
                    known = {**known, args[0]: args[1]}
                elif op == "s_and_b64" and args[:2] == ["vcc", "exec"]:
                    known = {**known, "vcc": known.get(args[2])}
                if op in ("s_branch", "s_endpgm", "s_setpc_b64") or op.startswith("s_cbranch"):
                    zero = {"0": True, "-1": False}.get(known.get("vcc")) if "vcc" in op else None
                    taken = None if zero is None else zero != op.endswith("nz")
                    if "branch" in op and taken is not False:
                        todo.append((labels[re.search(r"L\d+", args[-1]).group(0)], states + 1, known))
                    if not op.startswith("s_cbranch") or taken:
                        break
                states += int(args[0], 0) + 1 if op == "s_nop" else 1
                i += 1

    for i, (op, args) in enumerate(code):
        if product(op):
            result = registers(args[0])
            walk(i, BEHIND, lambda o, a: not product(o) and any(registers(x) & result for x in a))
        elif op.startswith("v_"):
            written = registers(args[0]) | (registers(args[1]) if op.startswith("v_swap") else set())
            if written:
                walk(i, BEFORE, lambda o, a: product(o) and any(registers(x) & written for x in a[1:4]))
    return found


MFMA = "v_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], a[8:11], v[0:3]"


@pytest.mark.parametrize("lines,wrong", [
    ([MFMA, "s_nop 9", "v_add_f32 v9, v1, v2"], 1),
    ([MFMA, "s_nop 10", "v_add_f32 v9, v1, v2"], 0),
    ([MFMA, MFMA, "s_nop 10", "v_mov_b32 v3, v9"], 0),
    ([MFMA, "s_nop 5", "v_mov_b32 v3, v9"], 1),
    (["v_mov_b32 v5, v9", "s_nop 0", MFMA], 1),
    (["v_mov_b32 v5, v9", "s_nop 1", MFMA], 0),
    (["v_accvgpr_write_b32 a8, v9", MFMA], 1),
    (["v_mov_b32 v12, v9", MFMA], 0),
    ([MFMA, "s_cbranch_scc1 L0", "s_endpgm", "<L0>:", "v_mov_b32 v3, v9"], 1),
    ([MFMA, "s_mov_b64 s[0:1], 0", "s_and_b64 vcc, exec, s[0:1]", "s_cbranch_vccz L0", "v_mov_b32 v3, v9", "<L0>:"], 0),
    ([MFMA, "s_mov_b64 s[0:1], -1", "s_and_b64 vcc, exec, s[0:1]", "s_cbranch_vccz L0", "v_mov_b32 v3, v9", "<L0>:"], 1),
    ([MFMA, "s_mov_b64 s[0:1], 0", "s_and_b64 vcc, exec, s[0:1]", "s_cbranch_vccnz L0", "s_endpgm", "<L0>:", "v_mov_b32 v3, v9"], 0),
    (["<L0>:", "v_mov_b32 v9, v1", "s_nop 15", MFMA, "s_cbranch_scc1 L0"], 1),
])
def test_the_walk_finds_what_is_too_close(lines, wrong):
    code, labels = functions("\n".join(["0000 <k>:"] + lines + ["s_endpgm"]))["k"]
    assert len(breaches(code, labels)) == wrong


@pytest.mark.skipif(not os.access(OBJDUMP, os.X_OK), reason="no disassembler here")
@pytest.mark.parametrize("kernel,instances", [("flash_prefill_wide_kernel", 6), ("gemm_prompt_kernel", 12)])
def test_products_written_by_hand_keep_their_distance(tmp_path, kernel, instances):
    lib = tmp_path / "lib.so"
    lib.symlink_to(build.ensure_built())
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, check=True, capture_output=True)
    image = next(p for p in sorted(tmp_path.glob("*" + build.ARCH)) if kernel.encode() in p.read_bytes())
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", "--symbolize-operands", str(image)],
                          check=True, capture_output=True, text=True).stdout
    mine = {n: f for n, f in functions(text).items() if kernel in n}
    assert len(mine) >= instances
    for name, (code, labels) in mine.items():
        assert sum(op.startswith("v_mfma") for op, _ in code) >= 32
        assert not breaches(code, labels), name
