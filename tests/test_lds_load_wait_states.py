"""Wait states in front of loads that write LDS.  Such a load takes its LDS address from M0 and may take
scalar operands; the hardware wants one instruction (or s_nop) between a scalar write of M0 and the load,
and five between a vector instruction's write of a scalar register and a memory instruction that reads
it.  The compiler sees to that for its own instructions but not for those inside inline assembly, where a load
that reads M0 too early puts its data into another place of LDS without any error.  So the device
assembly of every source with such loads is read here."""
import os
import re
import shutil
import subprocess

import pytest

from test_build_resources import CSRC, HIPCC

SOURCES = sorted(f for f in os.listdir(CSRC) if f.endswith(".hip")
                 and re.search(r"offen lds|load_lds", open(os.path.join(CSRC, f)).read()))
LDS_LOAD = re.compile(r"^(buffer_load_\w+ .*\blds\b|global_load_lds_\w+ .*)")
INSTRUCTION = re.compile(r"^\t([a-z]\w*(?: .*)?)$")


def scalar_registers(text):
    found = {"m0"} if re.search(r"\bm0\b", text) else set()
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        found |= {"s%d" % i for i in range(int(a), int(b) + 1)}
    return found | set(re.findall(r"\bs\d+\b", text)) | set(re.findall(r"\bvcc\b", text))


def violations(assembly):
    """(number of loads that write LDS, those with too few wait states before them)"""
    before, loads, bad = [], 0, []  # before: (wait states the instruction takes, text), newest last
    for line in assembly.splitlines():
        m = INSTRUCTION.match(line.split(";")[0].rstrip())
        if not m or m.group(1).startswith("."):
            continue
        text = m.group(1)
        if LDS_LOAD.match(text):
            loads += 1
            reads, passed = scalar_registers(text) | {"m0"}, 0
            for states, earlier in reversed(before):
                operands = earlier.split(" ", 1)[1] if " " in earlier else ""
                written = scalar_registers(operands.split(",")[0])
                need = 5 if earlier.startswith("v_") else 1 if "m0" in written else 0
                if passed < need and written & reads and not earlier.startswith(("s_cmp", "s_bitcmp")):
                    bad.append("%s | %s" % (earlier, text))
                passed += states
                if passed >= 5:
                    break
        nop = re.match(r"s_nop (\d+)", text)
        before = before[-5:] + [(int(nop.group(1)) + 1 if nop else 1, text)]
    return loads, bad


def test_the_check_itself():
    direct = "\ts_mov_b32 m0, s3\n\tbuffer_load_dwordx4 v1, s[4:7], s2 offen lds\n"
    assert violations(direct) == (1, ["s_mov_b32 m0, s3 | buffer_load_dwordx4 v1, s[4:7], s2 offen lds"])
    assert violations(direct.replace("\n\tb", "\n\ts_nop 0\n\tb")) == (1, [])
    assert violations(direct.replace("\n\tb", "\n\tv_add_u32_e32 v1, s3, v2\n\tb")) == (1, [])
    vector = "\tv_readfirstlane_b32 s6, v9\n\ts_nop %d\n\tbuffer_load_dwordx4 v1, s[4:7], s2 offen lds\n"
    assert len(violations(vector % 3)[1]) == 1 and violations(vector % 4) == (1, [])
    assert len(violations("\tv_readfirstlane_b32 m0, v9\n\ts_nop 0\n\tglobal_load_lds_dword v[2:3], off\n")[1]) == 1


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not found")
@pytest.mark.parametrize("source", SOURCES)
def test_loads_into_lds_wait_for_their_operands(source, tmp_path):
    out = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Xclang", "-target-feature",
                          "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", source, "-o", str(tmp_path / "out.s")],
                         cwd=CSRC, capture_output=True, text=True, timeout=600)
    assert out.returncode == 0, out.stderr[-2000:]
    assert "-Winline-asm" not in out.stderr, out.stderr[:2000]
    loads, bad = violations(open(tmp_path / "out.s").read())
    assert loads > 0
    assert not bad, "%d of %d loads: %s" % (len(bad), loads, bad[0])
