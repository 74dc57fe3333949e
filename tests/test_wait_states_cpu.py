"""Wait states that the compiler grants its own instructions, but not to inline assembly, hold in the library as built: every
kernel's instructions are walked backwards, over branches too, as far as the wait states reach."""
import collections
import os
import re
import shutil
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "fp-quant_amd", "fp_quant", "_lib", "libfpq_hip.so")
BIN = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def registers(operands):
    found = set()
    for kind, first, last, one in re.findall(r"\b([avs])(?:\[(\d+):(\d+)\]|(\d+)\b)", operands):
        found.update((kind, i) for i in (range(int(first), int(last) + 1) if first else (int(one),)))
    return found


def kernels(listing):
    """(name, [(opcode, operands)], {index: [indices of the branches that lead there]}) of llvm-objdump's output"""
    name, start, code, at, jumps = None, 0, [], {}, []
    for line in listing + ["0 <end>:"]:
        head = re.match(r"([0-9a-f]+) <(.*)>:", line)
        if head:
            if name:
                into = collections.defaultdict(list)
                for branch, target in jumps:
                    into[at[target]].append(branch)
                yield name, code, into
            name, start, code, at, jumps = head.group(2), int(head.group(1), 16), [], {}, []
        elif line.startswith("\t") and "//" in line:   # (the rest: zeros between kernels)
            text, _, note = line.partition("//")
            opcode, _, operands = text.strip().partition(" ")
            at[int(note.split(":")[0], 16)] = len(code)
            if "branch" in opcode:
                jumps.append((len(code), start + int(re.search(r"\+0x([0-9a-f]+)>", note).group(1), 16)))
            code.append((opcode, operands))


def writers_within(code, into, i, states, writes):
    """Instructions for which `writes` holds and after which fewer than `states` wait states pass before instruction i."""
    before = list(into[i])
    if i > 0 and code[i - 1][0] not in ("s_branch", "s_endpgm"):
        before.append(i - 1)
    for j in before:
        opcode, operands = code[j]
        if writes(opcode, operands):
            yield code[j]
        passed = int(operands, 0) + 1 if opcode == "s_nop" else 1
        if states > passed:
            yield from writers_within(code, into, j, states - passed, writes)


def matrix_operands_too_early(code, into):
    """A matrix instruction's registers, written by a vector instruction: two wait states."""
    for i, (opcode, operands) in enumerate(code):
        if opcode.startswith("v_mfma"):
            read = registers(operands.partition(",")[2])
            yield from writers_within(code, into, i, 2, lambda op, args: op.startswith("v_") and "mfma" not in op
                                      and bool(registers(args.split(",")[0]) & read))


def lds_address_too_early(code, into):
    """M0, from which a load to LDS takes its address: one wait state."""
    for i, (opcode, _) in enumerate(code):
        if opcode.startswith("global_load_lds"):
            yield from writers_within(code, into, i, 1, lambda op, args: args.split(",")[0].strip() == "m0")


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    if not os.path.exists(LIB) or not os.path.exists(os.path.join(BIN, "llvm-objdump")):
        pytest.skip("needs the built library and the compiler's llvm-objdump")
    where = tmp_path_factory.mktemp("code")
    shutil.copy(LIB, where / "lib.so")
    subprocess.run([os.path.join(BIN, "llvm-objdump"), "--offloading", "lib.so"], cwd=where, check=True, capture_output=True)
    return [k for f in sorted(os.listdir(where)) if "gfx950" in f for k in
            kernels(subprocess.run([os.path.join(BIN, "llvm-objdump"), "-d", "--no-show-raw-insn", f], cwd=where, check=True,
                                   capture_output=True, text=True).stdout.split("\n"))]


@pytest.mark.parametrize("rule,reads,at_least", [(matrix_operands_too_early, "v_mfma", 10000),
                                                 (lds_address_too_early, "global_load_lds", 1000)])
def test_wait_states(built, rule, reads, at_least):
    assert sum(op.startswith(reads) for _, code, _ in built for op, _ in code) >= at_least
    early = {name: found for name, code, into in built if (found := list(rule(code, into)))}
    assert not early


@pytest.mark.parametrize("gap,early", [([], True), (["s_waitcnt vmcnt(0)"], True), (["s_nop 0"], True), (["s_nop 1"], False),
                                       (["s_waitcnt vmcnt(0)", "v_mov_b32_e32 v1, v2"], False)])
def test_matrix_operands(gap, early):
    text = ["v_mov_b32_e32 v40, v2", *gap, "v_mfma_scale_f32_32x32x64_f8f6f4 v[2:17], v[18:21], v[22:25], v[2:17], v39, v40"]
    listing = ["0000000000000100 <kernel>:"] + [f"\t{t}  // {0x100 + 4 * i:012X}:" for i, t in enumerate(text)]
    (_, code, into), = kernels(listing)
    assert bool(list(matrix_operands_too_early(code, into))) == early
