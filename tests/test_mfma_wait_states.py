"""Results of the matrix cores that hand-written assembly reads.

The hardware does not hold back an instruction that reads an MFMA's result too early.  The compiler keeps the distance in
front of its own instructions, but it does not see what the assembly in the kernels reads, so the built code is looked at here:
no path from an MFMA to a store (or a DPP instruction) that only assembly makes has fewer wait states than the compiler keeps.
"""

import os
import re
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "swiftlm_amd", "lib", "libdflash_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
# what the compiler keeps between these and a reader of its own
WAIT_STATES = {"v_mfma_f32_16x16x4_f32": 10, "v_mfma_f32_16x16x16_bf16": 8, "v_mfma_f32_16x16x16_f16": 8, "v_mfma_f32_16x16x32_bf16": 8,
               "v_mfma_f32_16x16x32_f16": 8, "v_mfma_f32_32x32x16_bf16": 12, "v_mfma_f32_32x32x16_f16": 12}
LINE = re.compile(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):")
REGISTERS = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)")


def registers(text):
    return {(f, i) for f, a, b, c in REGISTERS.findall(text) for i in (range(int(a), int(b) + 1) if a else (int(c),))}


def only_assembly_makes(op, args):
    return (op.startswith("global_store") and args.endswith("sc0 sc1")) or (op.startswith("v_") and "row_newbcast" in args)


def functions(lines):
    name, code = None, []
    for line in lines:
        m = LINE.match(line)
        if m:
            code.append((m.group(1), m.group(2), int(m.group(3), 16)))
        elif line.endswith(">:"):
            if name:
                yield name, code
            name, code = line[line.index("<") + 1:-2], []
    if name:
        yield name, code


def too_early(code):
    """(MFMA, its address, reader, its address, wait states between them) for every reader that comes too early."""
    at = {address: i for i, (_, _, address) in enumerate(code)}
    for i, (mfma, args, address) in enumerate(code):
        if not mfma.startswith("v_mfma"):
            continue
        product, need = registers(args.split(",")[0]), WAIT_STATES[mfma]
        seen, paths = {}, [(i + 1, 0)]
        while paths:
            j, states = paths.pop()
            if j >= len(code) or states >= need or seen.get(j, need) <= states:
                continue
            seen[j] = states
            op, operands, here = code[j]
            if only_assembly_makes(op, operands) and registers(operands) & product:
                yield mfma, hex(address), op, hex(here), states
                continue
            if op == "s_endpgm":
                continue
            after = states + 1 + (int(operands) if op == "s_nop" else 0)
            if op == "s_branch" or op.startswith("s_cbranch"):
                words = int(operands.split()[0])
                target = here + 4 + 4 * (words - 65536 if words > 32767 else words)
                if target in at:
                    paths.append((at[target], after))
                if op == "s_branch":
                    continue
            paths.append((j + 1, after))


def test_no_assembly_reads_a_product_too_early(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    if not os.path.exists(LIB):
        import __graft_entry__

        __graft_entry__.build()
    lib = tmp_path / "lib.so"
    lib.write_bytes(open(LIB, "rb").read())
    subprocess.check_call([OBJDUMP, "--offloading", str(lib)], cwd=tmp_path, stdout=subprocess.DEVNULL)
    objects = sorted(tmp_path.glob("lib.so.*gfx950"))
    assert objects
    found, stores, kernels = [], 0, 0
    for path in objects:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], check=True, capture_output=True, text=True).stdout
        for name, code in functions(text.splitlines()):
            if any(op.startswith("v_mfma") for op, _, _ in code):
                kernels += 1
                stores += sum(only_assembly_makes(op, args) for op, args, _ in code)
                found += [(name, *early) for early in too_early(code)]
    assert kernels > 50 and stores > 100             # the listing is what this takes it for
    assert not found, found


@pytest.mark.parametrize("between,early", [(["s_nop 9"], False), (["s_nop 8"], True), (["s_nop 5", "s_barrier", "s_cbranch_scc1 1", "v_mov_b32_e32 v9, v8"], True),
                                           (["s_cbranch_scc0 1", "s_nop 9"], True), (["s_nop 6", "s_nop 2"], False)], ids=str)
def test_the_distance_is_counted(between, early):
    listing = ["v_mfma_f32_16x16x4_f32 v[2:5], v6, v7, v[2:5]", *between, "global_store_dwordx4 v[0:1], v[2:5], off sc0 sc1", "s_endpgm"]
    code = [(line.split()[0], line.partition(" ")[2], 4 * i) for i, line in enumerate(listing)]
    assert bool(list(too_early(code))) == early
