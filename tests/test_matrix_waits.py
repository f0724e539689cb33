"""No kernel reads what a matrix instruction makes before it is there.

The hardware does not wait for a matrix instruction's result where a vector or memory instruction reads or overwrites it: the compiler
leaves so many wait states in between.  It has left too few behind a branch that is taken (ROCm 7.2: the sums of ``delta_chain_kernel``,
when they were 32-bit and were added behind the branch over the next loads: 10 wait states where the branch falls through, 3 where it is
taken), so the built libraries' instructions are looked at: every way from a matrix instruction to the first use of its result."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from llama_cu_amd.kernels import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

# instruction: wait states before its result may be read or overwritten by anything but the next sum in the same registers; what the
# compiler leaves where no branch lies between, 4 and 8 passes of bfloat16, 8 of 32-bit and 16 of 64-bit
WAITS = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_32x32x16_bf16": 12, "v_mfma_f32_16x16x4_f32": 10, "v_mfma_f64_16x16x4_f64": 19}
LIBRARIES = ["attention_mfma", "attention_mfma_bias", "attention_mfma_cap", "decay_scan", "delta_rule", "gemm_mid", "gemm_skinny", "gemm_tiles", "gemm_wavek", "moe", "rglru"]

_REG = re.compile(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+))")
_LINE = re.compile(r"^\s+(\w+)\s*(.*?)\s*//\s*([0-9A-Fa-f]+):")
_HEAD = re.compile(r"^(?:([0-9a-fA-F]+) )?<(.+)>:$")
_GOAL = re.compile(r"<.+?(?:\+0x([0-9a-f]+))?>\s*$")


def registers(text):
    out = set()
    for kind, a, b, one in _REG.findall(text):
        out.update((kind, i) for i in (range(int(a), int(b) + 1) if a else [int(one)]))
    return out


def functions(listing):
    """``{name: [(operation, operands, number of the instruction a branch goes to or None)]}``"""
    found, name = {}, None
    for line in listing.splitlines():
        head = _HEAD.match(line.strip())
        if head:
            name = head.group(2)
            found[name] = []
            continue
        m = _LINE.match(line)
        if m and name is not None:
            goal = _GOAL.search(line) if m.group(1).startswith(("s_cbranch", "s_branch")) else None
            found[name].append((m.group(1), m.group(2), int(m.group(3), 16), int(goal.group(1) or "0", 16) if goal else None))
    for name, rows in found.items():
        at = {r[2]: i for i, r in enumerate(rows)}
        found[name] = [(op, args, at[rows[0][2] + goal] if goal is not None else None) for op, args, _, goal in rows]
    return found


def too_early(rows):
    """``(matrix instruction, its number, the use's number, wait states between)`` of every use that comes too early."""
    faults = []
    for k, (name, operands, _) in enumerate(rows):
        if "mfma" not in name:
            continue
        need, result = WAITS[name], registers(operands.split(",")[0])
        todo, seen = [(k + 1, 0)], {}
        while todo:
            i, waited = todo.pop()
            if i >= len(rows) or waited >= need or seen.get(i, need) <= waited:
                continue
            seen[i] = waited
            op, args, goal = rows[i]
            parts = args.split(",")
            if op in ("s_endpgm", "s_setpc_b64"):
                continue
            if goal is not None:
                todo.append((goal, waited + 1))
                if op != "s_branch":
                    todo.append((i + 1, waited + 1))
            elif op == "s_nop":
                todo.append((i + 1, waited + int(args, 0) + 1))
            elif op.startswith("s_"):
                todo.append((i + 1, waited + 1))
            elif "mfma" in op:
                if registers(",".join(parts[1:3])) & result:
                    faults.append((name, k, i, waited))
                elif not registers(parts[0] + "," + ",".join(parts[3:])) & result:      # (sums go on in the same registers: the hardware waits)
                    todo.append((i + 1, waited + 1))
            elif registers(args) & result:
                faults.append((name, k, i, waited))
            else:
                todo.append((i + 1, waited + 1))
    return faults


LOOP = """
<planted>:
\tv_mfma_f32_16x16x4_f32 v[0:3], v17, v83, v[0:3]            // 000000000100: 0
\ts_cbranch_scc1 3                                           // 000000000108: 0 <planted+0x{goal:x}>
\tglobal_load_dwordx4 v[6:9], v[4:5], off                    // 00000000010C: 0
\ts_nop {falls}                                                    // 000000000114: 0
\ts_nop {taken}                                                    // 000000000118: 0
\tv_add_f32_e32 v5, v3, v69                                  // 00000000011C: 0
\ts_endpgm                                                   // 000000000120: 0
"""


def test_a_use_behind_a_branch_is_found():
    use = lambda **kw: [f[2:] for f in too_early(functions(LOOP.format(**kw))["planted"])]
    assert use(goal=0x18, falls=5, taken=1) == [(5, 3)]              # taken: the branch and two; falling through: the branch, the load, six and two
    assert use(goal=0x18, falls=0, taken=8) == []
    assert use(goal=0x18, falls=0, taken=7) == [(5, 9)]
    assert use(goal=0x1C, falls=7, taken=0) == [(5, 1)]
    assert use(goal=0x20, falls=0, taken=0) == [(5, 4)]              # (taken, the result is not used)


def test_every_library_with_matrix_instructions_is_looked_at():
    kernels = os.path.dirname(build._sources("moe")[0])
    with_them = [n for n in build.KERNEL_LIBRARIES
                 if any("_mfma_" in open(p).read() for p in build._sources(n) + build._headers(n) if os.path.dirname(p) == kernels)]
    assert sorted(with_them) == sorted(LIBRARIES)


@pytest.mark.parametrize("name", LIBRARIES)
def test_results_of_matrix_instructions(name, tmp_path):
    if not os.path.isfile(OBJDUMP):
        pytest.skip("no llvm-objdump")
    built = build.build(name)
    copy = tmp_path / "library.so"
    copy.write_bytes(open(built, "rb").read())
    subprocess.run([OBJDUMP, "--offloading", copy.name], cwd=tmp_path, check=True, capture_output=True)
    device = [p for p in tmp_path.iterdir() if p.name.endswith("gfx950")]
    assert len(device) == 1
    listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(device[0])], check=True, capture_output=True, text=True).stdout
    count = 0
    for fn, rows in functions(listing).items():
        faults = too_early(rows)
        assert not faults, (fn, faults[:4])
        count += sum("mfma" in r[0] for r in rows)
    assert count > 0
