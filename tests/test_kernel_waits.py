"""Direct global->LDS loads and barriers in the built gfx950 code object.

A wave that moves data into LDS for its whole workgroup has to wait for those
loads before the barrier that publishes them; the compiler's own wait may come
later (where the wave itself reads the data).  This walks the control flow of
every kernel that uses such loads and requires that none is in flight at a
barrier."""
import os
import re
import subprocess

import pytest

import logicaffeine_amd as lgx

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
NONE = -1     # no direct load in flight; else the memory operations issued since the newest one


def kernels():
    if not os.path.exists(OBJDUMP) or not os.path.exists(lgx.HSACO_PATH):
        pytest.skip("no llvm-objdump or no built code object")
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", lgx.HSACO_PATH], check=True,
                          capture_output=True, text=True).stdout
    out, cur = {}, None
    for line in text.splitlines():
        head = re.match(r"^[0-9a-f]+ <(\S+)>:", line)
        if head:
            cur = out.setdefault(head.group(1), [])
        elif cur is not None and line.startswith("\t"):
            op, note = line.strip().split("//", 1)
            target = re.search(r"<\S+\+0x([0-9a-f]+)>", note)
            cur.append((int(re.search(r"([0-9A-F]{8,}):", note).group(1), 16), op.strip(),
                        int(target.group(1), 16) if target else None))
    return {k: v for k, v in out.items() if any("load_lds" in op for _, op, _ in v)}


def step(state, op):
    if "load_lds" in op:
        return 0
    wait = re.search(r"vmcnt\((\d+)\)", op) if op.startswith("s_waitcnt") else None
    if state != NONE and wait and state >= int(wait.group(1)):
        return NONE
    if state != NONE and op.startswith("s_waitcnt 0"):
        return NONE
    if state != NONE and re.match(r"(global|buffer|flat|scratch)_(load|store|atomic)", op):
        return state + 1
    return state


def unwaited_barriers(code):
    at = {addr: i for i, (addr, _, _) in enumerate(code)}
    states, work, found = {0: NONE}, [0], set()
    while work:
        i = work.pop()
        _, op, target = code[i]
        if op.startswith("s_barrier") and states[i] != NONE:
            found.add(i)
        out = step(states[i], op)
        nxt = [] if op.startswith(("s_branch", "s_endpgm")) else [i + 1]
        if op.startswith(("s_branch", "s_cbranch")) and target is not None:
            nxt.append(at[code[0][0] + target])
        for j in nxt:
            if j >= len(code):
                continue
            old = states.get(j)
            new = out if old in (None, NONE) else old if out == NONE else min(old, out)
            if new != old:
                states[j] = new
                work.append(j)
    return sorted(found)


def test_no_direct_load_is_in_flight_at_a_barrier():
    seen = kernels()
    assert any("attn_prefill_fast_d128" in k for k in seen)
    assert {k: b for k, b in ((k, unwaited_barriers(c)) for k, c in seen.items()) if b} == {}


def test_prefill_attention_v_loads_run_under_the_matrix_chains():
    """The exact prefill attention's V loads are in flight during products:
    the first stages' stand ahead of the score chain, every later one's is
    followed by products, not by a wait."""
    seen = {k: c for k, c in kernels().items() if re.match(r"lgx_k_attn_prefill\d*_d(64|128)_g\d$", k)}
    assert len(seen) >= 16
    for name, code in seen.items():
        ops = [op for _, op, _ in code]
        loads = [i for i, op in enumerate(ops) if "load_lds" in op]
        assert loads[0] < next(i for i, op in enumerate(ops) if op.startswith("v_mfma")), name
        for i in loads:
            state = 0                 # memory operations since the load
            for op in ops[i + 1:]:
                if op.startswith("v_mfma"):
                    break
                if re.match(r"(global|buffer|flat|scratch)_(load|store|atomic)", op):
                    state += 1
                wait = re.search(r"vmcnt\((\d+)\)", op)
                assert not (wait and state >= int(wait.group(1))), (name, i, op)


def test_kernels_keep_their_arrays_in_registers():
    """No kernel spills or indexes an array in scratch memory, except the two
    largest fast prefill attention forms (20 bytes, at 128 registers)."""
    if not os.path.exists(lgx.HSACO_PATH):
        pytest.skip("no built code object")
    readelf = os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf")
    notes = subprocess.run([readelf, "--notes", lgx.HSACO_PATH], check=True, capture_output=True, text=True).stdout
    size = dict(re.findall(r"\.name: +(lgx_k_\w+)\n\s+\.private_segment_fixed_size: (\d+)", notes))
    assert len(size) > 100
    kept = {f"lgx_k_attn_prefill_fast_d128_g{g}" for g in (7, 8)}
    assert {k: int(v) for k, v in size.items() if int(v) > (20 if k in kept else 0)} == {}
