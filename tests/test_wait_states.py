"""A mask or carry that a vector instruction writes to scalar registers (or vcc) is read by a vector instruction no sooner
than two wait states later.  The compiler sees to that between its own instructions; inside inline assembly, and for the
values that go in and out of it, it is ours to keep.  Checked on the machine code that this repository's build made."""
import os
import re
import subprocess

import pytest

from cachegen_amd.build import LIBRARY

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT = 2
# instructions whose second operand is a carry or mask that they write
CARRY_OUT = re.compile(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_mad_[ui]64|v_div_scale")
SCALAR_DESTINATION = re.compile(r"v_cmp|v_readfirstlane|v_readlane")


def scalar_registers(operand):
    m = re.match(r"(?:s\[(\d+):(\d+)\]|s(\d+)|(vcc))", operand.strip())
    if not m:
        return ()
    if m.group(4):
        return ("vcc",)
    return (int(m.group(3)),) if m.group(3) else range(int(m.group(1)), int(m.group(2)) + 1)


def early_readers(lines):
    """[(kernel, wait states between, writer, reader)] of a disassembly in program order."""
    out, kernel, written, t = [], None, {}, 0
    for line in lines:
        m = re.match(r"[0-9a-f]+ <(.*)>:", line)
        if m:
            kernel, written = m.group(1), {}
            continue
        name, _, rest = line.split("//")[0].strip().partition(" ")
        if name in ("s_branch", "s_setpc_b64", "s_endpgm"):     # what is written below is not what comes next
            written = {}
            continue
        if not rest:
            t += 1
            continue
        operands = rest.split(",")
        if name == "s_nop":
            t += int(operands[0], 0) + 1
            continue
        if name.startswith("v_"):
            if SCALAR_DESTINATION.match(name):
                destinations, sources = operands[:1], operands[1:]
            elif CARRY_OUT.match(name):
                destinations, sources = operands[1:2], operands[2:]
            else:
                destinations, sources = (), operands[1:]
            read = [written[r] for o in sources for r in scalar_registers(o) if r in written]
            if read and t - max(read)[0] - 1 < WAIT:
                out.append((kernel, t - max(read)[0] - 1, max(read)[1], line.split("//")[0].strip()))
            for r in (r for o in destinations for r in scalar_registers(o)):
                written[r] = (t, line.split("//")[0].strip())
        elif name.startswith("s_"):
            for r in scalar_registers(operands[0]):     # written by the scalar unit, whose results are waited for
                written.pop(r, None)
        t += 1
    return out


@pytest.mark.parametrize("code,early", [
    (["v_cmp_ge_u32_e64 s[2:3], v7, v15", "v_addc_co_u32_e64 v15, s[6:7], v3, v3, s[2:3]"], 1),
    (["v_cmp_ge_u32_e64 s[2:3], v7, v15", "s_nop 0", "v_addc_co_u32_e64 v15, s[6:7], v3, v3, s[2:3]"], 1),
    (["v_cmp_ge_u32_e64 s[2:3], v7, v15", "s_nop 1", "v_addc_co_u32_e64 v15, s[6:7], v3, v3, s[2:3]"], 0),
    (["v_add_co_u32_e32 v56, vcc, v56, v63", "v_mov_b32_e32 v1, v2", "v_addc_co_u32_e32 v57, vcc, 0, v57, vcc"], 1),
    (["v_add_co_u32_e32 v56, vcc, v56, v63", "v_mov_b32_e32 v1, v2", "v_mov_b32_e32 v1, v2", "v_addc_co_u32_e32 v57, vcc, 0, v57, vcc"], 0),
    (["v_cmp_ge_u32_e32 vcc, v7, v15", "s_mov_b64 vcc, -1", "v_addc_co_u32_e32 v57, vcc, 0, v57, vcc"], 0),
])
def test_the_check_itself(code, early):
    assert len(early_readers(["0 <k>:"] + code)) == early


def test_no_mask_is_read_early(tmp_path):
    link = tmp_path / "library.so"                        # the tool writes what it takes out beside what it reads
    os.symlink(LIBRARY, link)
    subprocess.run([OBJDUMP, "--offloading", str(link)], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    device = [f for f in os.listdir(tmp_path) if "gfx950" in f]
    assert len(device) == 1
    listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(tmp_path / device[0])], check=True, stdout=subprocess.PIPE, text=True).stdout
    lines = listing.splitlines()
    kernels = sum(line.endswith(">:") for line in lines)
    assert kernels > 100 and sum("v_addc_co_u32" in line for line in lines) > 100       # it is the library that was read
    early = early_readers(lines)
    assert not early, "%d readers, the first: %s" % (len(early), early[:3])
