"""Checks on the gfx950 code of the built library, read with llvm-objdump."""
import os
import re
import struct
import subprocess

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


# the opening of append_codes2 / append_int_codes: four compares, four selects, the first append
BLOCK = [re.compile(r"v_cmp_ge_(f32|i32)_e64 s\[")] * 4 + [re.compile(r"v_cndmask_b32_e64 ")] * 4 + [re.compile(r"v_addc_co_u32_e64 ")]


@pytest.mark.skipif(not (os.path.exists(LIB) and os.path.exists(OBJDUMP)), reason="needs the built library and llvm-objdump")
def test_assembly_waits_for_matrix_results(tmp_path):
    """The compiler puts wait states between a matrix instruction and vector instructions that read its result, but not
    for instructions inside assembly: wherever the code-appending block compares registers last written by a matrix
    instruction, the block has to be preceded by waits of its own."""
    blocks, fed, bad = 0, 0, []
    path = tmp_path / "code.o"
    for code in code_objects():
        path.write_bytes(code)
        if b"apnn_mfma_kernel" not in code and b"apnn_async_kernel" not in code and b"conv_i8_rows_kernel" not in code:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], check=True,
                              capture_output=True, text=True).stdout
        kernel, ins = "", []
        for line in text.splitlines():
            if line.endswith(">:"):
                kernel, ins = line, []
                continue
            s = line.split("//")[0].strip()
            if not s:
                continue
            ins.append(s)
            if not BLOCK[-1].match(s) or len(ins) < 9 or not all(p.match(i) for p, i in zip(BLOCK, ins[-9:])):
                continue
            blocks += 1
            wanted = set().union(*(registers(i.split(", ")[1]) for i in ins[-9:-5]))
            waited = False
            for i in reversed(ins[:-9]):
                waited = waited or i == "s_nop 15"
                op, _, rest = i.partition(" ")
                if not op.startswith("v_") and not op.startswith(("ds_read", "buffer_load", "global_load")):
                    continue
                wrote = registers(rest.split(", ")[0].strip()) & wanted
                if wrote and op.startswith("v_mfma"):
                    fed += 1
                    if not waited:
                        bad.append((kernel, ins[-9]))
                    break
                wanted -= wrote
                if not wanted:
                    break
    assert blocks > 100 and fed > 100, (blocks, fed)
    assert not bad, "%d of %d blocks read matrix results without waits: %s" % (len(bad), fed, bad[:4])
