"""The compiled direct filter gradient waits for its matrix products on every path.

A matrix instruction writes its result several issue slots after it starts and reads its addend while it
runs; whoever touches those registers earlier gets or leaves a wrong value, and nothing in the hardware
holds it back: the compiler has to put the wait there.  It does so inside a block of code and along most
branches, but a branch from a block that ends in matrix instructions to one with several ways in can come
without.  This walks all paths of the compiler's own listing."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "paralleltnnlayers_amd", "csrc")
PASSES = 4         # of v_mfma_f32_16x16x32_bf16, the one kind that the kernel has
RESULT = 8         # slots before its result may be read or overwritten: what the compiler itself leaves in a block
ADDEND = 3         # slots before its addend's registers may be overwritten


def _registers(operand):
    m = re.match(r"-?\|?v(?:\[(\d+):(\d+)\]|(\d+)\b)", operand.strip())
    if not m:
        return set()
    return set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}


def _kernels(listing):
    """(name, [(operation, operands) or (None, label)]) of each kernel."""
    name, code = None, []
    for line in listing.splitlines():
        line = line.split(";")[0].rstrip()
        label = re.match(r"([\w.$]+):", line)
        if label and label[1].startswith("_Z"):
            name, code = label[1], []
        elif label and label[1].startswith(".Lfunc_end") and name:
            yield name, code
            name = None
        elif label and name:
            code.append((None, label[1]))
        elif name and line.startswith("\t") and not line.strip().startswith("."):
            op, _, rest = line.strip().partition(" ") if "\t" not in line.strip() else line.strip().partition("\t")
            code.append((op, [a.strip() for a in rest.split(",")] if rest else []))


def too_early(code):
    """The first instruction that touches a matrix product or its addend too early, or None."""
    places = {label: i for i, (op, label) in enumerate(code) if op is None}
    for start, (op, args) in enumerate(code):
        if op is None or not op.startswith("v_mfma"):
            continue
        assert op == "v_mfma_f32_16x16x32_bf16", op
        result = _registers(args[0])
        addend = _registers(args[3]) - result
        todo, best = [(start + 1, 0, PASSES)], {}
        while todo:
            i, slots, free = todo.pop()                # free: when the matrix unit takes the next instruction
            while i < len(code) and slots < RESULT and best.get(i, 99) > slots:
                best[i] = slots
                op, args = code[i]
                i += 1
                if op is None:
                    continue
                if op == "s_endpgm":
                    break
                if op == "s_branch":
                    i = places[args[0]]
                elif op.startswith("s_cbranch"):
                    todo.append((places[args[0]], slots + 1, free))
                elif op == "s_nop":
                    slots += int(args[0], 0)
                elif op.startswith("v_mfma"):
                    if (_registers(args[1]) | _registers(args[2])) & result:
                        return f"{op} {args} after {slots} slots"
                    slots = max(slots, free - 1)
                    free = slots + PASSES
                    if _registers(args[0]) & result:   # (a chain: its successor is looked at on its own)
                        break
                elif op.startswith(("v_", "ds_", "buffer_", "global_", "flat_", "scratch_")):
                    stores = "store" in op or op.startswith("ds_write")
                    reads = set().union(*map(_registers, args if stores or op.startswith(("ds_", "v_fmac"))
                                             else args[1:]), set())
                    writes = set() if stores or not args else _registers(args[0])
                    if (reads | writes) & result or (op.startswith("v_") and slots < ADDEND and writes & addend):
                        return f"{op} {args} after {slots} slots"
                slots += 1
    return None


def _program(text):
    (_, code), = _kernels("_Zk:\n" + "".join(f"{l if l.startswith('.') else chr(9) + l}\n" for l in text) +
                          ".Lfunc_end0:\n")
    return code


MFMA = "v_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], v[12:15], v[4:7]"


@pytest.mark.parametrize("rest,early", [
    (["v_add_f32_e32 v20, v0, v21"], True), (["s_nop 6", "v_add_f32_e32 v20, v0, v21"], True),
    (["s_nop 7", "v_add_f32_e32 v20, v0, v21"], False), (["v_mov_b32_e32 v5, v20"], True),
    (["s_nop 2", "v_mov_b32_e32 v5, v20"], False), (["v_mov_b32_e32 v3, v20"], True),
    (["s_cbranch_vccnz .L1", "s_nop 7", ".L1:", "v_fmac_f32_e32 v0, v20, v21"], True),
    (["s_cbranch_vccnz .L1", "s_nop 7", ".L1:", "s_nop 6", "v_fmac_f32_e32 v0, v20, v21"], False),
    ([MFMA.replace("v[0:3]", "v[16:19]").replace("v[4:7]", "v[0:3]"), "v_mov_b32_e32 v4, v20"], False)])
def test_the_walk_itself(rest, early):
    assert bool(too_early(_program([MFMA] + rest + ["s_nop 15", "s_endpgm"]))) == early


def test_direct_filter_gradient(tmp_path):
    if not shutil.which("make") or not shutil.which("hipcc"):
        pytest.skip("no compiler for the kernels here")
    dry = subprocess.run(["make", "-C", CSRC, "-n", "-B", "bwd_filter_dense_direct.o"], check=True,
                         capture_output=True, text=True).stdout
    command = next(l for l in dry.splitlines() if "-c bwd_filter_dense_direct.hip" in l).split()
    listing = tmp_path / "direct.s"
    at = command.index("-c")
    subprocess.run(command[:at] + ["--offload-device-only", "-S", "bwd_filter_dense_direct.hip", "-o", str(listing)],
                   cwd=CSRC, check=True, capture_output=True)
    kernels = [(n, c) for n, c in _kernels(listing.read_text()) if "dense_direct_kernel" in n]
    assert kernels
    early = {n: e for n, e in ((n, too_early(c)) for n, c in kernels) if e}
    assert not early, early
