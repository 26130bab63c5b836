"""CPU-side check of the code generated for gfx950: tile copies (global_load_lds_*) against the reuse of the LDS they fill.

A copy is asynchronous and s_barrier does not wait for it, so LDS that copies fill may be written by other waves
only behind a barrier that every wave enters with its own copies landed.  The kernels turn their output rows through
the tile buffers: at the barrier in front of that no copy may be outstanding.  The copies are inline assembly, which
the compiler's own wait insertion does not see, and a copy that lands late is rare enough that results do not show
it; the instructions do."""
import os
import re
import shutil
import subprocess

import pytest

from mojodiffusion_amd import _lib

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


def _functions(lib, tmp):
    """{symbol: [(address, mnemonic, operands, branch target or None)]} of every gfx950 code object in `lib`."""
    copy = shutil.copy(lib, tmp)                    # (the bundles are written next to the input)
    subprocess.run([OBJDUMP, "--offloading", copy], check=True, stdout=subprocess.DEVNULL)
    out = {}
    for name in sorted(os.listdir(tmp)):
        if not name.endswith("gfx950"):
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", os.path.join(tmp, name)], check=True, capture_output=True, text=True).stdout
        base, code = {}, None
        for line in text.splitlines():
            m = re.match(r"([0-9a-f]+) <(\S+)>:$", line)
            if m:
                base[m[2]] = int(m[1], 16)
                code = out.setdefault(m[2], [])
                continue
            m = re.match(r"\s+(\S+)(.*?)\s*// ([0-9A-F]+):(?:.*<(\S+?)(?:\+0x([0-9a-f]+))?>)?", line)
            if m and code is not None:
                target = base[m[4]] + int(m[5] or "0", 16) if m[4] else None
                code.append((int(m[3], 16), m[1], m[2], target))
    return out


def _late_copies(code):
    """Addresses of the barriers that row stores follow without a further copy in between, and that can be reached
    with a copy outstanding."""
    index = {c[0]: i for i, c in enumerate(code)}

    def successors(i):
        _, op, _, target = code[i]
        if op == "s_endpgm":
            return []
        nxt = [index[target]] if op.startswith(("s_branch", "s_cbranch")) else []
        return nxt if op == "s_branch" else nxt + ([i + 1] if i + 1 < len(code) else [])

    def flood(start, stop):
        seen, todo = set(start), list(start)
        while todo:
            i = todo.pop()
            if not stop(i):
                for j in successors(i):
                    if j not in seen:
                        seen.add(j)
                        todo.append(j)
        return seen

    is_copy = lambda i: code[i][1].startswith("global_load_lds")
    landed = lambda i: code[i][1] == "s_waitcnt" and "vmcnt(0)" in code[i][2]
    copies = [i for i in range(len(code)) if is_copy(i)]
    outstanding = flood([j for i in copies for j in successors(i)], landed)
    bad = []
    for i, c in enumerate(code):
        if c[1] == "s_barrier" and i in outstanding:
            after = flood(successors(i), is_copy)
            if any(code[j][1] == "global_store_dwordx4" for j in after):
                bad.append(c[0])
    return len(copies), bad


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_no_copy_is_outstanding_when_the_tile_buffers_take_output_rows(tmp_path):
    """The main attention kernel, every instantiation.  (The short form and the backward end their copies by a wait
    for all of them on their last step only, a condition this path-blind search does not follow.)"""
    checked, late = 0, {}
    for name, code in _functions(_lib.LIB_PATH, tmp_path).items():
        if "sage_attn_kernel" in name:
            n, bad = _late_copies(code)
            assert n > 0 and any(c[1] == "global_store_dwordx4" for c in code), name
            checked += 1
            if bad:
                late[name] = ["%#x" % a for a in bad]
    assert checked >= 20 and not late, late


def test_the_check_sees_a_missing_wait():
    """The shape of the fault, and its mend, as a few instructions."""
    def code(wait):
        ops = [("global_load_lds_dwordx4", ""), wait, ("s_barrier", ""), ("ds_write_b64", ""), ("global_store_dwordx4", ""), ("s_endpgm", "")]
        return [(4 * i, op, args, None) for i, (op, args) in enumerate(ops)]
    assert _late_copies(code(("s_waitcnt", " lgkmcnt(0)"))) == (1, [8])
    assert _late_copies(code(("s_waitcnt", " vmcnt(2)"))) == (1, [8])
    assert _late_copies(code(("s_waitcnt", " vmcnt(0) lgkmcnt(0)"))) == (1, [])
