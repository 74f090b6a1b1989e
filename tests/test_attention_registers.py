"""The attention kernel keeps O and Q^T in accumulation registers that it names itself, and issues its matrix
instructions, tile copies and query loads from inline assembly, which the compiler does not look into.  What that relies
on is checked in the compiled code: the compiler uses no accumulation register of its own, nothing is spilled to memory,
and an address that a vector instruction has put into scalar registers is not read by a memory instruction within the
five wait states the hardware asks for."""
import os
import re
import subprocess

import pytest

from pbs_attn_amd import build


@pytest.fixture(scope="module", params=["pbs_attn.hip", "pbs_probe.hip"])
def kernels(request, tmp_path_factory):
    out = str(tmp_path_factory.mktemp("asm") / "k.s")
    cmd = [build._hipcc(), *build.DEVICE_FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, request.param), "-o", out]
    subprocess.run(cmd, check=True, capture_output=True)
    text = open(out).read()
    found = dict(re.findall(r"^(\S*(?:sparse_attn_kernel|tile_probe_kernel)\S*):.*?\n(.*?)s_endpgm", text, re.M | re.S))
    assert found
    return text, found


def test_accumulation_registers_are_touched_by_inline_assembly_only(kernels):
    for name, body in kernels[1].items():
        inside = False
        for line in body.splitlines():
            if "ASMSTART" in line or "ASMEND" in line:
                inside = "ASMSTART" in line
            elif not inside:
                assert not re.search(r"\ba\d|\ba\[|accvgpr", line.split(";")[0]), (name, line)


def test_nothing_is_spilled_to_memory(kernels):
    text, found = kernels
    for name, body in found.items():
        assert "scratch_" not in body and "buffer_store" not in body, name
        meta = text[text.index("amdhsa.kernels"):]
        entry = meta[meta.index(".name:           " + name):]
        assert int(re.search(r"\.private_segment_fixed_size: (\d+)", entry).group(1)) == 0, name
        assert int(re.search(r"\.vgpr_spill_count: (\d+)", entry).group(1)) == 0, name


def _scalar_regs(token):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", token)
    if m:
        return range(int(m[1]), int(m[2]) + 1)
    m = re.fullmatch(r"s(\d+)", token)
    return range(int(m[1]), int(m[1]) + 1) if m else ()


def test_scalar_addresses_written_by_vector_instructions_have_settled(kernels):
    for name, body in kernels[1].items():
        written, now = {}, 0          # scalar register -> when a vector instruction wrote it
        for line in body.splitlines():
            t = line.split(";")[0].replace(",", " ").split()
            if not t or t[0].startswith(".") or t[0].endswith(":"):
                continue
            now += 1 + (int(t[1]) if t[0] == "s_nop" else 0)
            if t[0].startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
                written.update({r: now for r in _scalar_regs(t[1])})
            elif t[0].startswith("s_") and len(t) > 1:
                for r in _scalar_regs(t[1]):
                    written.pop(r, None)
            elif t[0].startswith("global_"):
                for tok in t[1:]:
                    assert all(now - written.get(r, -9) > 5 for r in _scalar_regs(tok)), (name, line)
