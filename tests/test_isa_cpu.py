"""Checks on the gfx950 code of the built library, read with llvm-objdump."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "apnn-tc_amd", "lib", "libapnn_tc.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects():
    """The gfx950 code objects embedded in the library, one per translation unit."""
    with open(LIB, "rb") as f:
        data = f.read()
    at = data.find(MAGIC)
    while at >= 0:
        (entries,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(entries):
            offset, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


def registers(operand):
    """Vector registers named by an operand: v7 or v[4:19]."""
    m = re.fullmatch(r"v(\d+)", operand)
    if m:
        return {int(m.group(1))}
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", operand)
    return set(range(int(m.group(1)), int(m.group(2)) + 1)) if m else set()


def kernels():
    """(mangled name, instructions, their addresses) of every kernel of the library."""
    for code in code_objects():
        with tempfile.NamedTemporaryFile(suffix=".o") as f:
            f.write(code)
            f.flush()
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", f.name], check=True, capture_output=True, text=True).stdout
        name, ins, at = "", [], []
        for line in text.splitlines():
            if line.endswith(">:"):
                if ins:
                    yield name, ins, at
                name, ins, at = line, [], []
            elif "//" in line:
                s, _, where = line.partition("//")
                ins.append(s.strip())
                at.append(int(where.split(":")[0], 16))
        if ins:
            yield name, ins, at


def unsettled_results(ins, at):
    """Per instruction, the vector registers (bit masks) that a matrix instruction may have written last: (any, without
    a wait of sixteen states since), over all paths of the control flow."""
    index = {a: i for i, a in enumerate(at)}
    steps, nxt = [], []
    for i, s in enumerate(ins):
        op, _, rest = s.partition(" ")
        regs = 0
        if op.startswith(("v_", "ds_read", "buffer_load", "global_load")):
            for r in registers(rest.split(", ")[0].strip()):
                regs |= 1 << r
        steps.append((op.startswith("v_mfma"), s == "s_nop 15", regs))
        to = [i + 1] if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(ins) else []
        if op == "s_branch" or op.startswith("s_cbranch"):
            off = int(rest.split()[0])
            to.append(index[at[i] + 4 + 4 * (off - 65536 if off >= 32768 else off)])
        nxt.append(to)
    before = [(0, 0)] * len(ins)
    reached = [False] * len(ins)
    work = [0]
    reached[0] = True
    while work:
        i = work.pop()
        while True:
            any_, raw = before[i]
            mfma, wait, regs = steps[i]
            if wait:
                raw = 0
            any_, raw = (any_ | regs, raw | regs) if mfma else (any_ & ~regs, raw & ~regs)
            follow = None
            for j in nxt[i]:
                old = before[j]
                new = (old[0] | any_, old[1] | raw)
                if new != old or not reached[j]:
                    before[j], reached[j] = new, True
                    if follow is None:
                        follow = j
                    else:
                        work.append(j)
            if follow is None:
                break
            i = follow
    return before


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the built library and llvm-objdump")
def test_one_plane_convolutions_count_nothing():
    """Convolutions with one weight plane need no activation sums: symmetric weights are -1 / +1 operands, unsigned ones
    plain digits.  Their kernels hold no population count, also where the weight mode is a run-time value."""
    one_plane = re.compile(r"apnn_mfma_kernelILi1ELi\d+ELi1E(?:Li\d+E){5}Lb1E|apnn_async_kernelILi\d+ELi1E(?:Li\d+E){4}Lb1E")
    seen, bad = 0, []
    for name, ins, _ in kernels():
        if one_plane.search(name):
            seen += 1
            if any(i.startswith("v_bcnt_u32_b32") for i in ins):
                bad.append(name)
    assert seen > 40, seen
    assert not bad, "%d of %d kernels count activations: %s" % (len(bad), seen, bad[:3])


# the opening of append_codes2 / append_int_codes: four compares, four selects, the first append
BLOCK = [re.compile(r"v_cmp_ge_(f32|i32)_e64 s\[")] * 4 + [re.compile(r"v_cndmask_b32_e64 ")] * 4 + [re.compile(r"v_addc_co_u32_e64 ")]


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the built library and llvm-objdump")
def test_assembly_waits_for_matrix_results():
    """The compiler puts wait states between a matrix instruction and vector instructions that read its result, but not
    for instructions inside assembly: wherever the code-appending block compares registers last written by a matrix
    instruction, the block has to be preceded by waits of its own."""
    blocks, fed, bad = 0, 0, []
    for kernel, ins, at in kernels():
        found = [i for i in range(8, len(ins)) if BLOCK[-1].match(ins[i]) and all(p.match(s) for p, s in zip(BLOCK, ins[i - 8:i + 1]))]
        if not found:
            continue
        before = unsettled_results(ins, at)
        for i in found:
            blocks += 1
            wanted = 0
            for s in ins[i - 8:i - 4]:
                for r in registers(s.split(", ")[1]):
                    wanted |= 1 << r
            any_, raw = before[i - 8]
            fed += (any_ & wanted) != 0
            if raw & wanted:
                bad.append((kernel, ins[i - 8]))
    assert blocks > 100 and fed > 100, (blocks, fed)
    assert not bad, "%d of %d blocks read matrix results without waits: %s" % (len(bad), fed, bad[:4])
