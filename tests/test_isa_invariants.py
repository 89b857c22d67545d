"""Properties of the compiled gfx950 code that the kernels' speed rests on.

The device code of ``csrc/sas_capi.hip`` is compiled to assembly with the
library's own flags (about a minute) and checked for:

* no FLAT memory instruction in any kernel: a FLAT access counts on the LDS
  counter as well as the vector-memory one, so every LDS wait after it would
  also wait for the gathers in flight;
* no scratch: no kernel spills registers to memory;
* no ``s_waitcnt vmcnt(0)`` in the tile loop of the d_qk = 576 attention
  kernels: the loop keeps later tiles' DMAs in flight across its LDS reads,
  and a full vector-memory wait there (what the compiler emits when it cannot
  tell an LDS read from the tile ring's LDS-direct DMAs, e.g. once a second
  LDS object is in the kernel) serialises the gather with the MFMAs.
"""

from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from dsv4_planb_amd import build as B

SRC = os.path.join(B.CSRC, "sas_capi.hip")


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    if shutil.which(B.HIPCC) is None and not os.path.exists(B.HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("isa") / "sas_capi.s")
    r = subprocess.run([B.HIPCC, f"--offload-arch={B.ARCH}", *B.COMMON, *B.DEVICE_FLAGS,
                        "--cuda-device-only", "-S", SRC, "-o", out],
                       capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-2000:]
    with open(out) as f:
        return f.read().split("\n")


def _kernels(lines):
    """(symbol, body lines) of every kernel in the assembly."""
    out = []
    for i, l in enumerate(lines):
        m = re.match(r"^(_ZN3sas\w+): ; @", l)  # function labels (not data symbols)
        if m:
            end = next(j for j in range(i, len(lines)) if lines[j].startswith(".Lfunc_end"))
            out.append((m.group(1), lines[i:end]))
    return out


def _instr(l):
    s = l.strip()
    return s if l.startswith("\t") and s and not s.startswith((".", ";")) else None


def test_every_kernel_is_compiled(asm):
    names = [n for n, _ in _kernels(asm)]
    for k in ("plan_kernel", "resolve_kernel", "attend_kernel", "combine_kernel",
              "bwd_dq_kernel", "bwd_dkv_kernel"):
        assert any(k in n for n in names), k


def test_no_flat_memory_instructions(asm):
    bad = [(n[:60], _instr(l)) for n, body in _kernels(asm) for l in body
           if _instr(l) and re.match(r"flat_(load|store|atomic)", _instr(l))]
    assert not bad, bad[:5]


def test_no_scratch(asm):
    sizes = [int(l.split(":")[1]) for l in asm if l.strip().startswith(".private_segment_fixed_size:")]
    spills = [int(l.split(":")[1]) for l in asm if l.strip().startswith(".vgpr_spill_count:")]
    assert sizes and max(sizes) == 0
    assert spills and max(spills) == 0


def test_attention_tile_loop_keeps_dmas_in_flight(asm):
    checked = 0
    for name, body in _kernels(asm):
        if "attend_kernelILi576" not in name:
            continue
        labels = {}
        for i, l in enumerate(body):
            m = re.match(r"^(\.LBB\S+):", l)
            if m:
                labels[m.group(1)] = i
        loops = []
        for i, l in enumerate(body):
            m = re.match(r"\s+s_c?branch\w*\s+(\.LBB\S+)", l)
            if m and m.group(1) in labels and labels[m.group(1)] < i:
                a = labels[m.group(1)]
                loops.append((sum("v_mfma" in body[j] for j in range(a, i)), a, i))
        n_mfma, a, b = max(loops)
        assert n_mfma >= 50, (name[:60], n_mfma)
        waits = [body[j].strip() for j in range(a, b) if re.search(r"s_waitcnt vmcnt\(0\)", body[j])]
        assert not waits, (name[:60], waits[:3])
        checked += 1
    assert checked == 8  # {bf16, fp16} x {streaming, cached gather} x {16-bit, fp8 KV}


def test_narrow_tile_loop_keeps_dmas_in_flight(asm):
    """The two-wave attention kernel's loop: no full vector-memory wait either (a load
    copied where two ways through the loop join, or a global LDS-direct load the compiler
    counts, makes one)."""
    checked = 0
    for name, body in _kernels(asm):
        if "attend_narrow_kernelILi576" not in name:
            continue
        labels = {m.group(1): i for i, l in enumerate(body) if (m := re.match(r"^(\.LBB\S+):", l))}
        loops = []
        for i, l in enumerate(body):
            m = re.match(r"\s+s_c?branch\w*\s+(\.LBB\S+)", l)
            if m and m.group(1) in labels and labels[m.group(1)] < i:
                a = labels[m.group(1)]
                loops.append((sum("v_mfma" in body[j] for j in range(a, i)), a, i))
        # the shortest loop that holds a tile's 52 MFMAs (longer backward ranges also hold
        # the wait after the loop)
        _, a, b = min((e - s, s, e) for n, s, e in loops if n >= 52)
        waits = [body[j].strip() for j in range(a, b) if re.search(r"s_waitcnt vmcnt\(0\)", body[j])]
        assert not waits, (name[:60], waits[:3])
        checked += 1
    assert checked == 4


# scalar instructions that write SCC (moves, selects, multiplies, loads, waits and branches
# do not)
_WRITES_SCC = re.compile(r"\bs_(add|addc|sub|subb|absdiff|abs|min|max|and|or|xor|not|nand|nor|xnor|andn[12]|orn[12]|"
                         r"lsh[lr]\d?|ashr|bfe|bcnt\d|wqm|quadmask|cmp|cmpk|bitcmp\d|addk)_")


def test_assembly_that_writes_scc_says_so():
    """An asm statement whose instructions write SCC names it in its clobbers: otherwise the
    compiler may keep a comparison's result in SCC across the statement."""
    checked = 0
    for f in sorted(os.listdir(B.CSRC)):
        text = open(os.path.join(B.CSRC, f)).read() if f.endswith((".hip", ".h")) else ""
        for m in re.finditer(r"\basm\s+volatile\s*\(", text):
            depth, i = 1, m.end()
            while depth:
                depth += {"(": 1, ")": -1}.get(text[i], 0)
                i += 1
            stmt = text[m.start():i]
            checked += 1
            if _WRITES_SCC.search(stmt):
                assert '"scc"' in stmt, (f, text[:m.start()].count("\n") + 1)
    assert checked > 50
