"""Wait states inside inline assembly.

On gfx950 a vector instruction that reads a scalar register (vcc included) as data,
mask or carry must come at least two wait states after the vector instruction that
wrote it.  The compiler keeps the distance in the code it emits and does not look
inside an asm block, so the blocks of the sources that have vector instructions are
checked here, in the assembly the build's flags give: every vector instruction of
a block against every vector instruction before it."""
import os
import re
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "linbox_amd", "csrc")
WAIT = 2
SDST = re.compile(r"v_(add_co|addc_co|sub_co|subb_co|subrev_co|subbrev_co|mad_u64|mad_i64|div_scale)")


def scalars(op):
    """The scalar registers that an operand names."""
    op = op.strip().lstrip("-|").rstrip("|")
    if op == "vcc":
        return {"vcc_lo", "vcc_hi"}
    if op in ("vcc_lo", "vcc_hi") or re.fullmatch(r"s\d+", op):
        return {op}
    pair = re.fullmatch(r"s\[(\d+):(\d+)\]", op)
    return {"s%d" % i for i in range(int(pair.group(1)), int(pair.group(2)) + 1)} if pair else set()


def early_reads(lines):
    """(line number, text) of vector instructions in asm blocks that read a scalar
    register fewer than WAIT wait states after a vector instruction wrote it."""
    found, written, now, inside, seen = [], {}, 0, False, 0
    for no, line in enumerate(lines, 1):
        if "#ASMSTART" in line:
            inside = True
        elif "#ASMEND" in line:
            inside = False
        text = line.split(";")[0].split("//")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        name, _, rest = text.partition(" ")
        ops = [o for o in re.split(r",\s*(?![^\[]*\])", rest)] if rest else []
        if name == "s_nop":
            now += int(rest.strip(), 0) + 1
            continue
        if name.startswith("v_"):
            ndst = 2 if SDST.match(name) else 1
            if inside:
                seen += 1
                for op in ops[ndst:]:
                    if any(now - written.get(r, -9) - 1 < WAIT for r in scalars(op)):
                        found.append((no, text))
            for op in ops[:ndst]:
                for r in scalars(op):
                    written[r] = now
        now += 1
    return found, seen


def test_the_check_itself():
    block = ["\t;;#ASMSTART", "\tv_mad_u64_u32 v[2:3], vcc, v17, s12, v[2:3]", "\tv_addc_co_u32_e32 v64, vcc, 0, v64, vcc",
             "\t;;#ASMEND"]
    assert early_reads(block) == ([(3, "v_addc_co_u32_e32 v64, vcc, 0, v64, vcc")], 2)
    assert early_reads(block[:2] + ["\ts_nop 0"] + block[2:])[0]
    assert not early_reads(block[:2] + ["\ts_nop 1"] + block[2:])[0]
    assert not early_reads(block[:2] + ["\tv_mov_b32 v1, v2"] * 2 + block[2:])[0]
    assert not early_reads(block[1:])[0]  # outside a block
    before = ["\tv_readfirstlane_b32 s12, v9"] + block[:2] + ["\ts_nop 1"] + block[2:]
    assert early_reads(before)[0] == [(3, "v_mad_u64_u32 v[2:3], vcc, v17, s12, v[2:3]")]


def asm_sources():
    """Sources with inline vector assembly."""
    return [f for f in sorted(os.listdir(CSRC)) if f.endswith(".hip") and
            re.search(r'"v_|\\tv_', open(os.path.join(CSRC, f)).read())]


@pytest.mark.parametrize("source", asm_sources())
def test_asm_blocks_wait(source, tmp_path):
    sys.path.insert(0, ROOT)
    from linbox_amd import build_lib
    out = str(tmp_path / (source + ".s"))
    subprocess.run([build_lib.HIPCC] + build_lib.FLAGS + ["--cuda-device-only", "-S", os.path.join(CSRC, source),
                                                          "-o", out], check=True, capture_output=True)
    with open(out) as f:
        found, seen = early_reads(f.read().splitlines())
    assert seen > 0, "no vector instruction in an asm block: has the assembly's form changed?"
    assert not found, "%d of %d read a scalar register too early, first: %s" % (len(found), seen, found[:4])
