"""Scalar registers that the compiler keeps in lanes of a vector register, in
the simplex bookkeeping (advance_lane) of every build: no lane is read that has
no value on any path.  hipcc of ROCm 7.2 declares such a register without a
value where its first spill stands; inside a loop with several exits that loses
what earlier passes put there (the lanes that left by each exit), once the
register is given to other spills too.  Read from the assembly of this
library's own kernels, compiled here; needs no GPU."""
import concurrent.futures as cf
import glob
import os
import re
import subprocess

import pytest

from asteroid_amd import build

SOURCE = """
#include "ast_kernels.h"
namespace ast {
template <class CF>
__global__ void bookkeeping(const Machine<CF, (%s)>* m, LaneRegs<CF>* r, CF v) {
  advance_lane<CF, (%s)>(m[threadIdx.x], r[threadIdx.x], v, v > 0);
}
template __global__ void bookkeeping(const Machine<double, (%s)>*, LaneRegs<double>*, double);
template __global__ void bookkeeping(const Machine<float, (%s)>*, LaneRegs<float>*, float);
}
"""
DECLARED = re.compile(r"implicit-def: \$vgpr(\d+) : SGPR spill")
LANE = re.compile(r"(v_writelane_b32 v(\d+), \S+, (\d+)|v_readlane_b32 \S+, v(\d+), (\d+))$")
RELOAD = re.compile(r"scratch_load_dword v(\d+),.*Folded Reload")


def functions(text):
    """(name, lines) of each function of an assembly file."""
    for m in re.finditer(r"^(_Z\w+):[^\n]*\n(.*?)^\.Lfunc_end", text, re.M | re.S):
        yield m.group(1), m.group(2).split("\n")


def blocks(lines):
    """Basic blocks, their successors and, per block, what happens to spill
    registers: ("declare" | "write" | "read" | "reload", register, lane, line)."""
    out, label = [[]], {}
    for line in lines:
        m = re.match(r"(\.LBB\w+):", line)
        if m:
            out.append([])
            label[m.group(1)] = len(out) - 1
        out[-1].append(line)
        op = line.split(";")[0].split()
        if op and (op[0].startswith("s_cbranch") or op[0] in ("s_branch", "s_endpgm", "s_setpc_b64")):
            out.append([])
    after, events = [], []
    for k, block in enumerate(out):
        code = [line.split(";")[0].strip() for line in block]
        last = next((c.split() for c in reversed(code) if c), [""])
        nxt = [k + 1] if k + 1 < len(out) else []
        if last[0] == "s_branch":
            nxt = [label[last[1]]]
        elif last[0].startswith("s_cbranch"):
            nxt = nxt + [label[last[1]]]
        elif last[0] in ("s_endpgm", "s_setpc_b64"):
            nxt = []
        after.append(nxt)
        ev = []
        for line, c in zip(block, code):
            if m := DECLARED.search(line):
                ev.append(("declare", int(m.group(1)), 0, line))
            elif m := LANE.match(" ".join(c.split())):
                w, wl, r, rl = m.group(2, 3, 4, 5)
                ev.append(("write", int(w), int(wl), line) if w else ("read", int(r), int(rl), line))
            elif m := RELOAD.search(line):
                ev.append(("reload", int(m.group(1)), 0, line))
        events.append(ev)
    return after, events


def unwritten_reads(lines):
    """Reads of lanes that no path since the register's declaration has written."""
    after, events = blocks(lines)
    found = []

    def through(k, empty, report=False):
        empty = {r: set(lanes) for r, lanes in empty.items()}
        for what, reg, lane, line in events[k]:
            if what == "declare":
                empty[reg] = set(range(64))
            elif what == "reload":
                empty.pop(reg, None)
            elif what == "write":
                empty.get(reg, set()).discard(lane)
            elif report and lane in empty.get(reg, ()):
                found.append(line.strip())
        return empty

    at = [None] * len(events)  # lanes empty on every path to the block
    at[0], work = {}, [0]
    while work:
        k = work.pop()
        out = through(k, at[k])
        for n in after[k]:
            new = out if at[n] is None else {r: lanes & out.get(r, set()) for r, lanes in at[n].items()}
            if new != at[n]:
                at[n] = {r: set(lanes) for r, lanes in new.items()}
                work.append(n)
    for k in range(len(events)):
        if at[k] is not None:
            through(k, at[k], report=True)
    return found


def _variants():
    out = []
    for path in sorted(glob.glob(os.path.join(build.CSRC, "ast_k_*.hip"))):
        with open(path) as f:
            code = re.search(r"launch_variant<(.*?)>\(", f.read()).group(1)
        out.append(code.replace("VF_", "ast::VF_"))
    return out


def test_the_reader_finds_a_lost_lane():
    text = """_Zlost:
	s_mov_b32 s0, 0
.LBB0_1:
                                        ; implicit-def: $vgpr9 : SGPR spill to VGPR lane
	v_readlane_b32 s1, v9, 2
	s_or_b32 s1, s1, s0
	v_writelane_b32 v9, s1, 2
	v_readlane_b32 s2, v9, 2
	s_cbranch_execnz .LBB0_1
	v_readlane_b32 s3, v9, 2
	s_setpc_b64 s[30:31]
.Lfunc_end0:
"""
    assert [unwritten_reads(lines) for _, lines in functions(text)] == [["v_readlane_b32 s1, v9, 2"]]
    kept = text.replace("	s_mov_b32 s0, 0\n", "").replace(".LBB0_1:\n" + text.split("\n")[3] + "\n",
                                                             text.split("\n")[3] + "\n	v_writelane_b32 v9, s0, 2\n"
                                                             ".LBB0_1:\n")
    assert [unwritten_reads(lines) for _, lines in functions(kept)] == [[]]


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_no_lost_lane_in_any_build(tmp_path):
    variants = _variants()
    assert len(variants) == len(build.VARIANT_TUS)

    def one(k):
        src, out = tmp_path / f"b{k}.hip", tmp_path / f"b{k}.s"
        src.write_text(SOURCE.replace("%s", variants[k]))
        subprocess.run([build.HIPCC, "-S", "--cuda-device-only", "-w", *build.COMMON, *build.DEVICE, "-I", build.CSRC,
                        "-x", "hip", str(src), "-o", str(out)], check=True, capture_output=True)
        found = dict(functions(out.read_text()))
        assert sum("advance_lane" in name for name in found) == 2, variants[k]
        return {f"{variants[k]} {name}": r for name, lines in found.items() if (r := unwritten_reads(lines))}

    lost = {}
    with cf.ThreadPoolExecutor(8) as ex:
        for r in ex.map(one, range(len(variants))):
            lost.update(r)
    assert not lost
