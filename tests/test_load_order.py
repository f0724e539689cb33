"""Waits that count loads: the loads stand in the order and number that the counts take for granted.

The products whose rows reach LDS by loads of their own (``gemm_mid_ring_kernel``, ``gemm_tiles_kernel``) wait in front of a barrier until no more than N loads
are on their way.  That is a wait for a step's rows as long as exactly the later steps' loads were asked for behind them; a load that the compiler moves past another makes it a race
that tests on the GPU need not show.  So the built libraries' instructions are looked at: what is asked for between two barriers, in front of the loop and behind it."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from test_matrix_waits import OBJDUMP, functions

from llama_cu_amd.kernels import build


def kernels(name, tmp_path):
    """``{kernel: [(operation, operands, goal)]}`` of a built library."""
    if not os.path.isfile(OBJDUMP):
        pytest.skip("no llvm-objdump")
    copy = tmp_path / "library.so"
    copy.write_bytes(open(build.build(name), "rb").read())
    subprocess.run([OBJDUMP, "--offloading", copy.name], cwd=tmp_path, check=True, capture_output=True)
    device, = [p for p in tmp_path.iterdir() if p.name.endswith("gfx950")]
    return functions(subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(device)], check=True, capture_output=True, text=True).stdout)


def events(rows):
    """``(kind, what)`` of loads (``lds`` with the first register of their buffer, ``reg``), waits for loads (``wait`` with how many may be left) and barriers."""
    out = []
    for op, args, _ in rows:
        if op.startswith(("buffer_load", "global_load", "flat_load")):
            out.append(("lds", int(re.search(r"s\[(\d+):", args).group(1))) if re.search(r"\blds\b", args) else ("reg", None))
        elif op == "s_waitcnt" and "vmcnt" in args:
            out.append(("wait", int(re.search(r"vmcnt\((\d+)\)", args).group(1))))
        elif op == "s_barrier":
            out.append(("barrier", None))
    return out


def parts(rows):
    """The kernel's events in front of its loop, in it and behind it.  The loop: the one that loads to LDS and has barriers."""
    found = {(goal, i) for i, (_, _, goal) in enumerate(rows) if goal is not None and goal <= i
             and {"lds", "barrier"} <= {k for k, _ in events(rows[goal:i + 1])}}
    (first, last), = found
    return events(rows[:first]), events(rows[first:last + 1]), events(rows[last + 1:])


def waits_at_barriers(seen):
    """What may be left at each barrier: the wait that stands last in front of it."""
    out, last = [], None
    for kind, what in seen:
        if kind == "wait":
            last = what
        elif kind == "barrier":
            out.append(last)
            last = None
    return out


def loads(seen):
    return [e[0] for e in seen if e[0] in ("lds", "reg")]


def check_ring(rows, mt, swiglu, d, waves, tiles):
    """``gemm_mid_ring_kernel``: each of D steps waits for all but the W of D - 1 steps and the X of D - 2, then asks for a later step's X, then its W."""
    w, x = 4 * (2 if swiglu else tiles), (mt + 1) // 2 if waves == 8 else mt
    front, loop, behind = parts(rows)
    left = (d - 1) * w + (d - 2) * x
    step = [("wait", left), ("barrier", None)] + ["lds"] * x + ["reg"] * w
    assert [e if e[0] in ("wait", "barrier") else e[0] for e in loop] == step * d
    begin = (["reg"] * w + ["lds"] * x) * (d - 1) + ["reg"] * w
    assert loads(front)[-len(begin):] == begin and "lds" not in loads(front)[:-len(begin)]
    assert loads(behind) == [] and waits_at_barriers(behind) == [(d - 1 - i) * w + (d - 2 - i) * x for i in range(d - 1)]


def check_tiles(rows, ft, tt, wf, wt, sf, st):
    """``gemm_tiles_kernel``: a step waits for all but what the later of its two loads were followed by, then asks for tokens, then for features."""
    f, t = 32 * ft * wf // 8 // (wf * wt), 32 * tt * wt // 8 // (wf * wt)
    front, loop, behind = parts(rows)
    left = (f if sf > st else 0) + (st - 2) * (f + t)
    tokens = next(what for kind, what in loop if kind == "lds")
    features, = {what for kind, what in loop if kind == "lds"} - {tokens}
    turn = [("lds", tokens)] * t + [("lds", features)] * f
    assert loop == [("wait", left), ("barrier", None)] + turn
    assert [e for e in front if e[0] == "lds"] == [("lds", features)] * f * (sf - st) + turn * (st - 1)
    assert loads(behind) == [] and waits_at_barriers(behind) == [0]


def numbers(name, pattern):
    return [int(x) for x in re.search(pattern, name).groups()]


RING, TILES = r"ring_kernelILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E", r"GtShapeILi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)ELi(\d+)E"


def ring_of(name):
    mt, epilogue, d, waves, tiles = numbers(name, RING)
    return mt, epilogue == 2, d, waves, tiles


def test_rows_that_share_lds(tmp_path):
    found = {n: r for n, r in kernels("gemm_mid", tmp_path).items() if "gemm_mid_ring_kernel" in n}
    assert len(found) >= 17
    for name, rows in found.items():
        assert numbers(name, RING)[1] in (1, 2)
        check_ring(rows, *ring_of(name))


def test_many_rows_in_tiles(tmp_path):
    found = {n: r for n, r in kernels("gemm_tiles", tmp_path).items() if "gemm_tiles_kernel" in n}
    assert len(found) == 9
    for name, rows in found.items():
        check_tiles(rows, *numbers(name, TILES))


def places(rows, what):
    """Where in the loop the loads to LDS (``lds``), other loads (``reg``) and counting waits in front of a barrier stand."""
    (first, last), = {(goal, i) for i, (_, _, goal) in enumerate(rows) if goal is not None and goal <= i and {"lds", "barrier"} <= {k for k, _ in events(rows[goal:i + 1])}}
    return [i for i in range(first, last + 1) if (events(rows[i:i + 1]) or [(None, None)])[0][0] == what]


def test_planted_mistakes_are_found(tmp_path):
    """A load of W in front of the last one of X, a count that is one too high, a load that is gone, tokens behind features: in a copy of the listing."""
    name, rows = next((n, r) for n, r in kernels("gemm_mid", tmp_path).items() if "ring_kernelILi4ELi1ELi3ELi4ELi1E" in n)
    check = lambda r: check_ring(r, *ring_of(name))
    check(rows)

    def swapped(r, i, j):
        r = list(r)
        r[i], r[j] = r[j], r[i]
        return r
    lds, reg, waits = (places(rows, k) for k in ("lds", "reg", "wait"))
    counted = lambda r, i: r[:i] + [(r[i][0], re.sub(r"vmcnt\((\d+)\)", lambda m: f"vmcnt({int(m.group(1)) + 1})", r[i][1]), r[i][2])] + r[i + 1:]
    for bad in (swapped(rows, lds[3], reg[0]), counted(rows, waits[0]), rows[:lds[0]] + [("s_nop", "0", None)] + rows[lds[0] + 1:], rows[:reg[-1]] + [("s_nop", "0", None)] + rows[reg[-1] + 1:]):
        with pytest.raises(AssertionError):
            check(bad)
    (tmp_path / "tiles").mkdir()
    name, rows = next((n, r) for n, r in kernels("gemm_tiles", tmp_path / "tiles").items() if "GtShapeILi4ELi2ELi2ELi4ELi3ELi2E" in n)
    check = lambda r: check_tiles(r, *numbers(name, TILES))
    check(rows)
    lds, waits = places(rows, "lds"), places(rows, "wait")
    for bad in (swapped(rows, lds[0], lds[-1]), counted(rows, waits[0]), rows[:lds[0]] + [("s_nop", "0", None)] + rows[lds[0] + 1:]):
        with pytest.raises(AssertionError):
            check(bad)
