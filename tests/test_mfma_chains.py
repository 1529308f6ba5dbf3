"""No kernel of the built library hands an accumulator from a 16x16x16 to a 16x16x32 bf16 matrix product, or back, without
enough wait states in between: the hardware does not wait and the compiler does not know (mm2 and settle in
csrc/hdla_common.cuh).  Reads the library's own machine code; on the CPU."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from hdla_hip import _lib

OBJDUMP = shutil.which("llvm-objdump", path=os.pathsep.join(["/opt/rocm/llvm/bin", os.environ.get("PATH", "")]))
WAIT = 6            # wait states below which a pair is reported; 5 were enough where it was measured
MFMA = re.compile(r"v_mfma_f32_16x16x(16|32)_bf16 v\[(\d+):(\d+)\], \S+ \S+ (?:v\[(\d+):(\d+)\]|\S+)")


def pairs_too_close(lines):
    """(line number, text) of products whose accumulator a product of the other shape wrote less than WAIT wait states before."""
    found, recent, now = [], [], 0
    for no, ln in enumerate(lines):
        ln = ln.split("//")[0].strip()
        if not ln or ln.endswith(":"):
            continue
        now += 1
        m = re.match(r"s_nop (\d+|0x[0-9a-f]+)", ln)
        if m:
            now += int(m[1], 0)
        m = MFMA.match(ln)
        if not m:
            continue
        if m[4]:
            c0, c1 = int(m[4]), int(m[5])
            if any(now - at <= WAIT and shape != m[1] and d0 <= c1 and c0 <= d1 for at, shape, d0, d1 in recent):
                found.append((no, ln))
        recent = [r for r in recent if now - r[0] <= WAIT] + [(now, m[1], int(m[2]), int(m[3]))]
    return found


def code_objects(path):
    """The gfx950 code objects in a library built by hipcc: entries of its offload bundles."""
    blob, magic, at = open(path, "rb").read(), b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        n, = struct.unpack_from("<Q", blob, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + ln]
            pos += 24 + ln
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at += len(magic)


def test_the_check_finds_a_planted_pair():
    x16, x32 = "v_mfma_f32_16x16x16_bf16 v[0:3], v[8:9], v[10:11], ", "v_mfma_f32_16x16x32_bf16 v[4:7], v[8:11], v[12:15], "
    assert pairs_too_close([x16 + "0", x32 + "v[0:3]"])
    assert pairs_too_close([x32 + "0", "s_nop 1", x16 + "v[4:7]"])
    assert not pairs_too_close([x16 + "0", "s_nop 7", x32 + "v[0:3]"])
    assert not pairs_too_close([x16 + "0", x16 + "v[0:3]", x32 + "v[4:7]"])


@pytest.mark.skipif(OBJDUMP is None, reason="no llvm-objdump")
def test_no_accumulator_changes_product_shape_without_a_wait(tmp_path):
    path = _lib.lib_path()
    if not os.path.exists(path):
        pytest.skip("the library is not built")
    seen, bad = 0, []
    for i, code in enumerate(code_objects(path)):
        f = tmp_path / ("%d.o" % i)
        f.write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(f)], check=True, capture_output=True, text=True).stdout
        lines = text.splitlines()
        seen += sum("16x16x32_bf16" in ln for ln in lines)
        bad += [(i, no, ln) for no, ln in pairs_too_close(lines)]
    assert seen > 0, "no 16x16x32 product found: the disassembly was not read"
    assert not bad, bad[:5]
