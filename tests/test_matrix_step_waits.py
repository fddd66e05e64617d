"""No instruction of the built kernels reads a matrix step's result too early.

A vector or memory instruction that reads the result of a matrix step needs
wait states after it (18 for the FP64 16 x 16 x 4 step, 10 for the FP32 one and
for the bfloat16 16 x 16 x 32 one, whatever of it the reader needs), which the
compiler inserts.  Where the reader follows behind a branch around a short block
it has left them out, and the results were wrong.  This walks every path from
every matrix step in the objects that the library was linked from."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BUILD = os.path.join(ROOT, "libflame_amd", "_build")
LLVM = "/opt/rocm/llvm/bin/"
TARGET = "hipv4-amdgcn-amd-amdhsa--gfx950"
NEED = {"v_mfma_f64_16x16x4_f64": 18, "v_mfma_f32_16x16x4_f32": 10,
        "v_mfma_f32_16x16x32_bf16": 10}
OBJECTS = sorted(f[:-6] for f in os.listdir(BUILD)
                 if f.endswith(".hip.o") and f != "fla_hip_runtime.hip.o") if os.path.isdir(BUILD) else []
# the first operand is read too, or is the only one read
READS_FIRST = ("global_store", "buffer_store", "scratch_store", "flat_store", "ds_write",
               "global_atomic", "v_fmac", "v_readlane", "v_readfirstlane", "v_permlane",
               "v_swap", "v_cmpx")
NO_RESULT = READS_FIRST[:6]


def registers(operand):
    m = re.match(r"-?\|?v\[(\d+):(\d+)\]", operand) or re.match(r"-?\|?v(\d+)", operand)
    if not m:
        return frozenset()
    return frozenset(range(int(m[1]), int(m[m.lastindex]) + 1))


def instructions(text):
    """[(address, name, operand registers, operands)] and the index of each address."""
    symbols, ins = {}, []
    for line in text.splitlines():
        m = re.match(r"([0-9a-f]+) <(.+)>:", line)
        if m:
            symbols[m[2]] = int(m[1], 16)
            continue
        m = re.match(r"\s+(\w+)\s*(.*?)\s*// ([0-9A-F]+):[^<]*(?:<(.+?)(?:\+0x([0-9a-f]+))?>)?$", line)
        if not m:
            continue
        ops = [o.strip() for o in m[2].split(",")] if m[2] else []
        target = symbols.get(m[4], 0) + int(m[5] or "0", 16) if m[4] else None
        ins.append((int(m[3], 16), m[1], [registers(o) for o in ops], ops, target))
    return ins, {x[0]: k for k, x in enumerate(ins)}


def early_reads(text):
    ins, at = instructions(text)
    found = set()
    for start, (_, name, regs, _, _) in enumerate(ins):
        if not name.startswith("v_mfma"):
            continue
        need, seen = NEED[name], {}
        paths = [(start + 1, 0, regs[0])]
        while paths:
            k, waited, live = paths.pop()
            while k < len(ins) and waited < need and live:
                if seen.get((k, live), need) <= waited:
                    break
                seen[k, live] = waited
                _, op, r, ops, target = ins[k]
                if op in ("s_endpgm", "s_setpc_b64", "s_swappc_b64"):
                    break
                if op.startswith("v_mfma"):
                    if (r[1] | r[2]) & live:
                        found.add((start, k))
                        break
                    live = live - r[0]  # accumulated or overwritten by the matrix unit, in order
                else:
                    first = 0 if op.startswith(READS_FIRST) else 1
                    if any(x & live for x in r[first:]):
                        found.add((start, k))
                        break
                    if op.startswith("v_") and r:
                        live = live - r[0]
                waited += int(ops[0]) + 1 if op == "s_nop" else 1
                if op == "s_branch":
                    k = at[target]
                    continue
                if op.startswith("s_cbranch"):
                    paths.append((at[target], waited, live))
                k += 1
    return [(ins[a][0], ins[a][1], hex(ins[b][0]), ins[b][1], ins[b][3]) for a, b in sorted(found)]


def disassembly(name, tmp):
    fat, code = os.path.join(tmp, "fat"), os.path.join(tmp, "code")
    run = lambda *a: subprocess.run([LLVM + a[0], *a[1:]], check=True, capture_output=True, text=True).stdout  # noqa: E731,E501
    run("llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, os.path.join(BUILD, name + ".hip.o"),
        os.path.join(tmp, "copy"))
    run("clang-offload-bundler", "--unbundle", "--type=o", "--input=" + fat, "--targets=" + TARGET,
        "--output=" + code)
    return run("llvm-objdump", "-d", "--no-show-raw-insn", code)


def test_a_read_behind_a_branch_is_found():
    text = """
0000000000001000 <k>:
\tv_mfma_f32_16x16x4_f32 v[4:7], v0, v1, v[4:7]             // 000000001000: 00
\ts_cbranch_scc0 2                                          // 000000001008: 00 <k+0x14>
\ts_nop 7                                                   // 00000000100C: 00
\ts_nop 7                                                   // 000000001010: 00
\tv_add_f32_e32 v2, v7, v3                                  // 000000001014: 00
\ts_endpgm                                                  // 000000001018: 00
"""
    assert len(early_reads(text)) == 1
    assert not early_reads(text.replace("s_cbranch_scc0 2 ", "s_nop 9          "))
    assert not early_reads(text.replace("v2, v7, v3", "v2, v8, v3"))


@pytest.mark.skipif(not OBJECTS, reason="the library's objects are not here")
@pytest.mark.parametrize("name", OBJECTS)
def test_no_early_reads(name, tmp_path):
    text = disassembly(name, str(tmp_path))
    assert "s_endpgm" in text or "v_mfma" not in text
    assert early_reads(text) == []
