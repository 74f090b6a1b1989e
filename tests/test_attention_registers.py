"""The attention kernel keeps O and Q^T in accumulation registers that it names itself, and issues its matrix
instructions, tile copies and query loads from inline assembly, which the compiler does not look into.  What that relies
on is checked in the compiled code: the compiler uses no accumulation register of its own, nothing is spilled to memory,
results of matrix instructions are given their time, an address that a vector instruction has put into scalar registers is not read by a memory instruction within the
five wait states the hardware asks for; and a load into an accumulation register is awaited before the register is read."""
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
    found = dict(re.findall(r"^(\S*(?:sparse_attn_kernel|tile_probe_kernel)\S*):.*?\n(.*?)^\.Lfunc_end", text, re.M | re.S))
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


def _acc_regs(token):
    m = re.fullmatch(r"a\[(\w+)(?::(\w+))?\]", token) or re.fullmatch(r"a(\d+)()", token)
    if not m:
        return ()
    lo = int(m[1], 0)
    return range(lo, int(m[2], 0) + 1 if m[2] else lo + 1)


def _unfinished_reads(body):
    """Instructions that may meet an accumulation register whose load has not been awaited, over every path through the
    branches of `body`.  Vector memory operations complete in order, so `s_waitcnt vmcnt(n)` completes a load that at least
    n younger ones follow on the path: the state is, per register with a load on its way, the smallest such number."""
    code, at = [], {}
    for line in body.splitlines():
        t = line.split(";")[0].strip()
        if re.fullmatch(r"\S+:", t):
            at[t[:-1]] = len(code)
        elif t and not t.startswith("."):
            code.append(t.replace(",", " ").split())
    assert not any(t[0].startswith(("s_swappc", "s_call", "s_cbranch_g", "s_cbranch_join")) for t in code)
    heads = set(at.values())
    states, todo, bad = {0: {}}, [0], set()

    def flow(to, state):
        known = states.get(to)
        merged = dict(state) if known is None else {r: min(state.get(r, 99), known.get(r, 99)) for r in {*state, *known}}
        if merged != known:
            states[to] = merged
            todo.append(to)

    while todo:
        i = head = todo.pop()
        state = dict(states[i])
        while i < len(code):
            t = code[i]
            op = t[0]
            load = op.startswith("global_load") and "lds" not in op
            regs = {r for tok in t[1:] for r in _acc_regs(tok)}
            if not load and regs & state.keys():
                bad.add(" ".join(t))
            if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
                state = {r: n + 1 for r, n in state.items()}
            if load:
                state.update(dict.fromkeys(regs, 0))
            if op == "s_waitcnt":
                m = re.search(r"vmcnt\((\d+)\)", " ".join(t))
                if m:
                    state = {r: n for r, n in state.items() if n < int(m[1])}
            # where its block leaves the lane mask alone, some lane is always there
            some_lane = op.startswith("s_cbranch_exec") and not any("exec" in tok for u in code[head:i] for tok in u[1:])
            if op.startswith(("s_branch", "s_cbranch")) and not (some_lane and op == "s_cbranch_execz"):
                flow(at[t[1]], state)
            if some_lane and op == "s_cbranch_execnz":
                break
            if op == "s_setpc_b64":   # a branch out of a conditional one's reach: getpc, add (label - .Lpost_getpc), addc, setpc
                flow(at[re.search(r"\((\.LBB\w+)-\.Lpost_getpc", " ".join(code[i - 2]))[1]], state)
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                break
            i += 1
            if i in heads:
                flow(i, state)
                break
    return sorted(bad)


def test_the_walk_finds_a_missing_wait():
    load, copy = "global_load_dwordx4 a[0xc0:0xc3], v[0:1], off\n", "global_load_lds_dwordx4 v0, s[0:1]\n"
    use, loop = "v_accvgpr_mov_b32 a[0x80], a[0xc3]\n", "s_cbranch_scc1 .L1\n"
    assert _unfinished_reads(load + use)
    assert _unfinished_reads(load + "s_waitcnt lgkmcnt(0)\n" + use)
    assert not _unfinished_reads(load + "s_waitcnt vmcnt(0) lgkmcnt(0)\n" + use)
    assert _unfinished_reads(load + copy + "s_waitcnt vmcnt(2)\n" + use)
    assert not _unfinished_reads(load + copy + copy + "s_waitcnt vmcnt(2)\n" + use)
    assert _unfinished_reads(load + loop + copy + ".L1:\ns_waitcnt vmcnt(1)\n" + use)               # the path without the copy
    assert _unfinished_reads(".L1:\nv_mfma_f32 v[0:3], v[4:7], a[192:195], 0\n" + load + loop)      # round the loop
    assert not _unfinished_reads(".L1:\ns_waitcnt vmcnt(0)\nv_mfma_f32 v[0:3], v[4:7], a[192:195], 0\n" + load + loop)
    far = "s_getpc_b64 s[0:1]\n.Lpost_getpc0:\ns_add_u32 s0, s0, (.LBB1_2-.Lpost_getpc0)&4294967295\n" \
          "s_addc_u32 s1, s1, (.LBB1_2-.Lpost_getpc0)>>32\ns_setpc_b64 s[0:1]\ns_waitcnt vmcnt(0)\n.LBB1_2:\n"
    assert _unfinished_reads(load + far + use)


def test_loads_into_accumulation_registers_are_awaited_on_every_path(kernels):
    """The compiler does not know of loads issued in inline assembly, and the hardware does not hold a reader up."""
    for name, body in kernels[1].items():
        assert re.search(r"global_load_dwordx4 a\[", body), name
        assert not _unfinished_reads(body), name


def _vector_regs(token):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", token) or re.fullmatch(r"[-|]*v(\d+)()\|?", token)
    return range(int(m[1]), int(m[2] or m[1]) + 1) if m else ()


def test_results_of_matrix_instructions_have_settled(kernels):
    """The result of a matrix instruction may be touched by other instructions 11 wait states after it, what a vector instruction
    wrote may be read by a matrix instruction 3 states after it.  The compiler sees to that for its own matrix
    instructions only.  In order of the code; a matrix instruction counts as the four states for which it holds the pipe."""
    for name, body in kernels[1].items():
        issued, written, now = {}, {}, 0
        for line in body.splitlines():
            t = line.split(";")[0].replace(",", " ").split()
            if not t or t[0].startswith(".") or t[0].endswith(":"):
                continue
            if t[0].startswith("v_mfma"):
                assert all(now - written.get(r, -9) >= 3 for tok in t[2:4] for r in _vector_regs(tok)), (name, line)
                issued.update(dict.fromkeys(_vector_regs(t[1]), now))
                now += 4
                continue
            assert all(now - issued.get(r, -99) > 11 for tok in t[1:] for r in _vector_regs(tok)), (name, line)
            if t[0].startswith("v_"):
                for r in _vector_regs(t[1]):
                    written[r] = now
                    issued.pop(r, None)
            now += 1 + (int(t[1]) if t[0] == "s_nop" else 0)
