"""Hazards the compiler does not pad around inline asm, checked in the gfx950
assembly of every kernel source.

The kernels issue their DMA, Q and some store instructions as inline asm.
The compiler inserts the wait states the hardware needs between ordinary
instructions, but it does not look inside an asm statement, so two hazards
can reach the GPU unpadded (both were seen there as wrong, run-to-run
varying results):

* a VALU instruction writes an SGPR (v_readlane restoring a spilled SGPR,
  v_readfirstlane, a VOP3 compare) and a vector memory instruction in asm
  reads it fewer than 5 wait states later: the load or store uses a stale
  descriptor or offset word;
* a vector memory store of more than 8 bytes in asm, after which the
  compiler rewrites the store's data VGPRs fewer than 2 wait states later:
  the store reads its data after issue and sends the new values.

A third check covers the padding the tree kernels carry by hand: a
ds_read_b64_tr_b16 that refills an MFMA's A or B operand registers fewer
than 16 wait states after that MFMA issued corrupted the MFMA's operand
(wrong, run-to-run varying outputs), so every such read must come at least
16 wait states after the MFMA.

The check compiles each source to assembly (hipcc -S, the library's flags)
and scans it. CPU only; skipped where hipcc is absent.
"""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "quail_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["-O3", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", "-Wno-inline-asm", "--cuda-device-only", "-S"]
SOURCES = {"attention.hip": [], "gemm_fp8.hip": [], "fused.hip": ["-ffp-contract=off"],
           "runtime.hip": []}


def _regs(text, prefix):
    """Register numbers of one kind (s or v) named in an operand string."""
    out = set()
    for m in re.finditer(prefix + r"\[(\d+):(\d+)\]", text):
        out.update(range(int(m.group(1)), int(m.group(2)) + 1))
    for m in re.finditer(r"\b" + prefix + r"(\d+)\b", text):
        out.add(int(m.group(1)))
    return out


def _wait_states(ins):
    m = re.match(r"s_nop\s+(\d+)", ins)
    return int(m.group(1)) + 1 if m else 1


def scan(asm_text):
    """Findings of both hazards in one assembly file (a list of strings)."""
    found = []
    lines = asm_text.split("\n")
    in_asm = False
    history = []  # (instruction, sgprs written by a VALU op)
    pending_stores = []  # (line, data vgprs, wait states since)
    func = "?"
    for n, raw in enumerate(lines, 1):
        s = raw.strip()
        if re.match(r"^_Z\w+:", s):
            func, history, pending_stores = s.split(":")[0], [], []
            continue
        if s.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if s.startswith(";;#ASMEND"):
            in_asm = False
            continue
        if not s or s.startswith(";") or s.startswith(".") or s.endswith(":"):
            continue
        ins = s.split(";")[0].strip()
        op = ins.split()[0]
        args = ins[len(op):]
        dst = args.split(",")[0] if "," in args else args
        # a write to the data of an asm store still being read
        writes_v = _regs(dst, "v") if op.startswith(("v_", "ds_read", "buffer_load",
                                                      "global_load")) else set()
        for line0, data, ws in pending_stores:
            if ws < 2 and writes_v & data:
                found.append(f"{func}: line {n} `{ins}` rewrites the data of the asm store "
                             f"at line {line0} after {ws} wait states")
        pending_stores = [(l0, d, w + _wait_states(ins)) for l0, d, w in pending_stores
                          if w + _wait_states(ins) < 2]
        if in_asm and op.startswith(("buffer_", "global_")):
            used = _regs(args, "s")
            ws = 0
            for prev, written in reversed(history):
                if written & used:
                    if ws < 5:
                        found.append(f"{func}: line {n} `{ins}` reads s{sorted(written & used)} "
                                     f"{ws} wait states after `{prev}`")
                    break
                ws += _wait_states(prev)
                if ws >= 5:
                    break
            if op.startswith("buffer_store_dwordx") or op.startswith("global_store_dwordx"):
                width = int(re.search(r"dwordx(\d)", op).group(1))
                if width > 2:
                    pending_stores.append((n, _regs(args.split(",")[0], "v"), 0))
        valu_sgpr = set()
        if op.startswith("v_") and ("readlane" in op or "readfirstlane" in op
                                    or (op.startswith("v_cmp") and "_e64" in op)):
            valu_sgpr = _regs(dst, "s")
        history.append((ins, valu_sgpr))
        history = history[-16:]
    return found


def scan_tr_reads(asm_text, need=16):
    """ds_read_b64_tr_b16 writes into a recent MFMA's A/B operand registers."""
    found = []
    lines = [l.strip() for l in asm_text.split("\n")]
    func = "?"
    for n, s in enumerate(lines):
        if re.match(r"^_Z\w+:", s):
            func = s.split(":")[0]
        if not s.startswith("v_mfma"):
            continue
        ops = [o.strip() for o in s.split(";")[0].split(None, 1)[1].split(",")]
        srcs = _regs(ops[1], "v") | _regs(ops[2], "v")
        ws = 0
        for m in range(n + 1, len(lines)):
            t = lines[m]
            if not t or t.startswith(";") or t.startswith(".") or t.endswith(":"):
                if t.endswith(":") and not t.startswith(";"):
                    break  # a label: control flow joins here; stop the window
                continue
            if t.startswith("s_endpgm") or re.match(r"s_(c?branch|setpc)", t):
                break
            op = t.split()[0]
            if op.startswith("ds_read_b64_tr_b16"):
                dst = t.split()[1].rstrip(",")
                if _regs(dst, "v") & srcs:
                    found.append(f"{func}: line {m + 1} `{t}` refills an operand of the MFMA at "
                                 f"line {n + 1} after {ws} wait states")
            ws += _wait_states(op if op != "s_nop" else t)
            if ws >= need:
                break
    return found


def test_the_scanner_flags_both_hazards():
    # a stale SGPR read and a store whose data is rewritten at once
    bad = "\n".join([
        "_Zkernel:",
        "\tv_readlane_b32 s7, v164, 3",
        ";;#ASMSTART",
        "\tbuffer_load_dwordx4 v[82:85], v3, s[4:7], 0 offen",
        ";;#ASMEND",
        ";;#ASMSTART",
        "\tbuffer_store_dwordx4 v[2:5], v11, s[68:71], 0 offen",
        ";;#ASMEND",
        "\tv_lshl_add_u32 v2, v11, 7, v9",
    ])
    found = scan(bad)
    assert len(found) == 2, found
    good = "\n".join([
        "_Zkernel:",
        "\tv_readlane_b32 s7, v164, 3",
        ";;#ASMSTART",
        "\ts_nop 4",
        "\tbuffer_load_dwordx4 v[82:85], v3, s[4:7], 0 offen",
        ";;#ASMEND",
        ";;#ASMSTART",
        "\tbuffer_store_dwordx4 v[2:5], v11, s[68:71], 0 offen",
        "\ts_nop 1",
        ";;#ASMEND",
        "\tv_lshl_add_u32 v2, v11, 7, v9",
    ])
    assert scan(good) == []


def test_the_transposed_read_check_flags_an_early_refill():
    bad = "\n".join([
        "_Zkernel:",
        "\tv_mfma_f32_32x32x16_bf16 v[146:161], v[4:7], v[186:189], v[146:161]",
        "\ts_nop 7",
        "\tds_read_b64_tr_b16 v[4:5], v3 offset:512",
    ])
    assert len(scan_tr_reads(bad)) == 1
    good = bad.replace("\ts_nop 7", "\ts_nop 7\n\ts_nop 7")
    assert scan_tr_reads(good) == []


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC),
                    reason="hipcc is not installed")
@pytest.mark.parametrize("source", sorted(SOURCES))
def test_no_unpadded_inline_asm_hazard(source, tmp_path):
    out = tmp_path / (source + ".s")
    cmd = [HIPCC, *FLAGS, *SOURCES[source], os.path.join(CSRC, source), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, cwd=CSRC, timeout=600)
    text = out.read_text()
    found = scan(text) + scan_tr_reads(text)
    assert not found, "\n".join(found[:10])


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC),
                    reason="hipcc is not installed")
@pytest.mark.parametrize("source", ["attention.hip", "gemm_fp8.hip"])
def test_no_kernel_with_asm_loads_spills_vgprs(source, tmp_path):
    """The compiler takes the outputs of a load in an asm statement as written
    at once. Spilled, such a register is stored while its load is in flight and
    then reused, and the load lands on the new value: an address, once, and the
    access faulted. These sources keep asm loads in flight across steps, so
    none of their kernels may use scratch memory."""
    out = tmp_path / (source + ".s")
    cmd = [HIPCC, *FLAGS, os.path.join(CSRC, source), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, cwd=CSRC, timeout=600)
    text = out.read_text()
    spills = re.findall(r"\.name:\s+(_Z\w+)(?:(?!\.name:).)*?\.vgpr_spill_count:\s+(\d+)", text, re.S)
    assert spills and not [s for s in spills if s[1] != "0"], spills
