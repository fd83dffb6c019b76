"""Instructions written by hand keep the wait states that the compiler gives its own (CPU: the sources compiled to gfx950
assembly with the library's own flags).  A vector instruction that reads a scalar register needs two of them behind the vector
instruction that wrote it -- a comparison, an addition with carry, a lane read; the hardware does not wait by itself and
the compiler looks at no instruction inside an asm block."""
import os
import re
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "triton-hub_amd", "csrc")
WAIT_STATES = 2
SECOND_RESULT = re.compile(r"v_(add|addc|sub|subb|subrev|subbrev)_co_|v_div_scale_|v_mad_[ui]64_")   # its carry or mask


def scalar_registers(operand):
    """The scalar registers of one operand of an instruction."""
    found = {r for r in ("vcc",) if re.search(r"\bvcc\b", operand)}
    for first, last in re.findall(r"\bs\[(\d+):(\d+)\]", operand):
        found |= {f"s{n}" for n in range(int(first), int(last) + 1)}
    return found | set(re.findall(r"\bs\d+\b", operand))


def hazards(assembly):
    """Pairs of lines with too few wait states between them."""
    bad, written, state = [], {}, 0          # register -> (wait states passed when it was written, line)
    for number, line in enumerate(assembly.splitlines(), 1):
        text = line.split(";")[0].strip()
        if not line.startswith("\t") or not re.match(r"[a-z]\w*(\s|$)", text):       # labels, directives, comments
            continue
        name, _, rest = text.partition(" ")
        operands = rest.split(",")
        if name.startswith("v_"):
            results = 2 if SECOND_RESULT.match(name) else 1
            for register in set().union(*map(scalar_registers, operands[results:])):
                if register in written and state - written[register][0] < WAIT_STATES:
                    bad.append((written[register][1], f"{number}: {text}"))
            for register in set().union(*map(scalar_registers, operands[:results])):
                written[register] = (state + 1, f"{number}: {text}")
        elif name.startswith("s_"):
            for register in scalar_registers(operands[0]):      # a scalar result: the hardware waits for it
                written.pop(register, None)
        state += int(operands[0], 0) + 1 if name == "s_nop" else 1
    return bad


def test_rule_on_written_out_pairs():
    compare, read = "\tv_cmp_gt_u32_e64 s[4:5], s1, v2\n", "\tv_cndmask_b32_e64 v3, v4, 0, s[4:5]\n"
    other = "\tv_add_u32_e32 v7, v8, v9\n"
    assert hazards(compare + read) and hazards(compare + other + read) and hazards(compare + "\ts_nop 0\n" + read)
    assert not hazards(compare + "\ts_nop 1\n" + read) and not hazards(compare + other + other + read)
    assert not hazards(compare + "\ts_mov_b64 s[4:5], 0\n" + read)
    assert hazards("\tv_mad_u64_u32 v[2:3], s[6:7], v1, v1, 0\n" + "\tv_mul_f32_e32 v3, s7, v3\n")
    assert not hazards("\tv_mad_u64_u32 v[2:3], s[6:7], v1, v1, 0\n" + "\tv_mad_u64_u32 v[4:5], s[6:7], v1, v1, 0\n")


@pytest.mark.parametrize("unit", ["thn_dropout"])          # the sources with instructions in asm blocks
def test_scalar_results_are_read_late_enough(unit, tmp_path):
    target = tmp_path / f"{unit}.o"
    subprocess.check_call(["make", "-s", "-C", CSRC, f"OBJDIR={tmp_path}", "EXTRA=--offload-device-only -S", str(target)])
    assembly = target.read_text()
    assert "v_addc_co_u32_e64" in assembly and assembly.count(".amdhsa_kernel") >= 20
    assert hazards(assembly) == []


def test_other_sources_have_no_instructions_in_asm_blocks():
    blocks = {}
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".h", ".hip")):
            text = re.sub(r"//.*", "", open(os.path.join(CSRC, name)).read())
            blocks[name] = [b for b in re.findall(r"\basm\s*(?:volatile\s*)?\(\s*\"([^\"]*)\"", text) if b]
    assert {name for name, found in blocks.items() if found} == {"thn_dropout.h"}
