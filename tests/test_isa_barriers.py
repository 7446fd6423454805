"""The built gfx950 code at its barriers: a barrier that frees an LDS buffer for the next loads must not be passed while this
wave still reads it. A fragment read that is queued when the wave passes s_barrier can be overtaken by another wave's load into
that buffer (stale operands now and then, with no error), so every kernel that fills LDS by direct loads waits for its reads
(lgkmcnt) first. Checked on the disassembly of libhexanima_hip.so, over every path through each kernel."""
import os
import re
import shutil
import subprocess

import pytest

from hexanima_amd import hip

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


def _kernels(pattern, tmp):
    """{symbol: [(address, instruction, branch target or None)]} of the library's kernels whose symbol matches"""
    lib = os.path.join(tmp, "lib.so")
    shutil.copy(hip.LIB_PATH, lib)
    subprocess.run([OBJDUMP, "--offloading", lib], capture_output=True, check=True, cwd=tmp)
    out = {}
    for f in sorted(os.listdir(tmp)):
        if "gfx950" not in f:
            continue
        syms = subprocess.run([OBJDUMP, "-t", os.path.join(tmp, f)], capture_output=True, text=True, check=True).stdout
        names = [l.split()[-1] for l in syms.splitlines() if " .text" in l and re.search(pattern, l)]
        if not names:
            continue
        txt = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + ",".join(names), os.path.join(tmp, f)],
                             capture_output=True, text=True, check=True).stdout
        cur = None
        for l in txt.splitlines():
            h = re.match(r"^[0-9a-f]+ <(\S+)>:$", l)
            if h:
                cur = out.setdefault(h[1], [])
                continue
            m = re.match(r"^\s+(.*?)\s*// ([0-9A-F]+):", l)
            if m and cur is not None:
                at = int(m[2], 16)
                b = re.match(r"s_c?branch\S*\s+(\d+)$", m[1])
                simm = int(b[1]) if b else None
                cur.append((at, m[1], None if simm is None else at + 4 + 4 * (simm - 65536 if simm >= 32768 else simm)))
    return out


def _reads_at_barriers(ins):
    """[(index of s_barrier, most LDS reads outstanding there on any path)]"""
    index = {at: k for k, (at, _, _) in enumerate(ins)}
    state, work = [-1] * len(ins), [0]
    state[0] = 0
    while work:
        k = work.pop()
        n, (_, s, target) = state[k], ins[k]
        op = s.split()[0]
        if op.startswith("ds_read"):
            n = min(n + 1, 64)
        elif op == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", s)
            n = min(n, int(m[1])) if m else n
        nxt = [] if op in ("s_endpgm", "s_branch") else [k + 1]
        if target is not None:
            nxt.append(index[target])
        for q in nxt:
            if q < len(ins) and state[q] < n:
                state[q] = n
                work.append(q)
    return [(k, state[k]) for k, (_, s, _) in enumerate(ins) if s.startswith("s_barrier") and state[k] >= 0]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    # (the attention kernels, and one GEMM of each loop form and weight format)
    return _kernels(r"attn_kernel|attn_short|gemm_xattn|gemm_skinny_kernelILi64|gemm_pair_kernelILi128ELi128|"
                    r"gemm_kernelILi(256ELi256|192ELi128|128ELi128|64ELi64)E", str(tmp_path_factory.mktemp("isa")))


def test_no_barrier_is_passed_with_a_fragment_read_in_flight(kernels):
    assert len(kernels) > 20
    bad = {n: [r for r in _reads_at_barriers(ins) if r[1] > 0] for n, ins in kernels.items()}
    assert not {n: r for n, r in bad.items() if r}


def test_three_phase_attention_waits_at_its_barriers_itself(kernels):
    """The three-phase loop frees a buffer one barrier after its last read: its barriers carry their own lgkmcnt(0), so that
    this does not rest on where the compiler puts the last MFMAs of a phase."""
    three = {n: ins for n, ins in kernels.items() if "attn_kernelILi6E" in n}
    assert len(three) == 2
    for n, ins in three.items():
        bars = [k for k, (_, s, _) in enumerate(ins) if s.startswith("s_barrier")]
        own = [k for k in bars if any("lgkmcnt(0)" in s for _, s, _ in ins[max(0, k - 3):k])]
        # all but the first (no LDS read before it) and the two of the merge of the key halves
        assert set(bars[1:-2]) <= set(own) and len(bars) >= 8, (n, len(bars), len(own))
