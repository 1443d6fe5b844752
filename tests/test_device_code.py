"""The machine code that the build makes of the kernels, where inline assembly
and hardware rules meet (no GPU: the library's own code objects are listed with
the toolchain's disassembler)."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import old_fmm_bem_amd as F

OBJDUMP = next((p for p in ("/opt/rocm/llvm/bin/llvm-objdump", shutil.which("llvm-objdump")) if p and os.path.exists(p)),
               None)
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """the gfx950 code objects of an offload bundle sequence"""
    at = blob.find(MAGIC)
    while at >= 0:
        pos, out = at + len(MAGIC) + 8, []
        for _ in range(struct.unpack_from("<Q", blob, at + len(MAGIC))[0]):
            off, size, ln = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + ln]
            pos += 24 + ln
            if b"gfx950" in name and size:
                out.append(blob[at + off:at + off + size])
        yield from out
        at = blob.find(MAGIC, pos)


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """{kernel symbol: [instruction, ...]} of every kernel"""
    if OBJDUMP is None:
        pytest.skip("no llvm-objdump")
    with open(F.library_path(), "rb") as f:
        blob = f.read()
    d, kernels = tmp_path_factory.mktemp("code"), {}
    for k, obj in enumerate(_code_objects(blob)):
        path = str(d / f"{k}.co")
        with open(path, "wb") as f:
            f.write(obj)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", path], check=True,
                              capture_output=True, text=True).stdout
        cur = None
        for line in text.splitlines():
            m = re.match(r"<(\w+)>:|[0-9a-f]+ <(\w+)>:", line)
            if m:
                cur = kernels.setdefault(m.group(1) or m.group(2), [])
            elif cur is not None and line.strip():
                cur.append(line.split("//")[0].strip())
    assert any("k_m2l_o" in k for k in kernels)
    return kernels


def test_lds_copies_wait_for_m0(listing):
    """A scalar write of M0 needs one wait state before a copy into LDS that
    takes its address from it (any instruction in between is one)."""
    copies, bad = 0, []
    for name, code in listing.items():
        for prev, ins in zip(code, code[1:]):
            op = ins.split()[0]
            if "load_lds" in op or (op.startswith("buffer_load") and " lds" in ins):
                copies += 1
                if re.match(r"s_\w+ m0,", prev):
                    bad.append((name, prev, ins))
    assert copies > 0
    assert not bad, (len(bad), copies, bad[:3])


def _span(operand):
    """(file, first, last) of a register operand, None for a constant"""
    m = re.match(r"([av])(?:\[(\d+):(\d+)\]|(\d+))$", operand.strip().split(" ")[0])
    return m and (m.group(1), int(m.group(2) or m.group(4)), int(m.group(3) or m.group(4)))


def test_fp64_mfma_outputs_leave_their_operands_alone(listing):
    """v_mfma_f64_16x16x4 writes its output while it still reads its operands:
    they must not share registers."""
    seen, bad = set(), []
    for name, code in listing.items():
        for ins in code:
            if not ins.startswith("v_mfma_f64_16x16x4"):
                continue
            seen.add(name)
            d, a, b = (_span(o) for o in ins.split(None, 1)[1].split(",")[:3])
            if any(o and o[0] == d[0] and o[1] <= d[2] and d[1] <= o[2] for o in (a, b)):
                bad.append((name, ins))
    assert any("k_m2l_of" in k for k in seen) and any("k_translate_mfma" in k for k in seen)
    assert not bad, bad[:3]
