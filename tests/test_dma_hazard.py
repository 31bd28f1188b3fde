"""The wait states in front of the inline-assembly DMA, in the compiled kernels.

A vector memory instruction may read an SGPR that a vector instruction wrote
(v_readfirstlane, v_readlane, a compare) only five wait states later.  The
compiler keeps that for its own instructions and not for inline assembly, so
a source base that comes straight from a v_readfirstlane lets the DMA read
from a wrong address.  The DMA helpers therefore take a DmaSrc only, whose
maker waits; these tests compile every source the way the Makefile does, look
the AMD assembly over for such a pair, and need no GPU.
"""

import re
import shutil

import pytest

from conftest import HIPCC, assemble, build_recipes

WAIT_STATES = 5
pytestmark = pytest.mark.skipif(not shutil.which(HIPCC), reason="hipcc not found")


def _sgprs(operands):
    regs = {int(n) for n in re.findall(r"\bs(\d+)\b", operands)}
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", operands):
        regs |= set(range(int(lo), int(hi) + 1))
    return regs | {name for name in ("vcc", "m0") if re.search(rf"\b{name}", operands)}


def _parse(asm):
    """Per function: instructions as (name, SGPRs a vector instruction writes,
    SGPRs a vector memory instruction reads, wait states, line) and, for each,
    the instructions that can come before it."""
    functions, instrs, labels, branches, pending = [], [], {}, [], []
    for number, line in enumerate(asm.splitlines(), 1):
        text = line.split(";")[0].strip()
        label = re.match(r"([.\w$]+):", text)
        if label:
            if not label[1].startswith("."):
                instrs, labels, branches = [], {}, []
                functions.append((label[1], instrs, labels, branches))
            labels[label[1]] = len(instrs)
            continue
        if not text or text.startswith("."):
            continue
        op, _, args = text.partition(" ")
        first = args.split(",")[0]
        writes, reads, states = set(), set(), 1
        if op == "s_nop":
            states = int(args, 0) + 1
        elif op.startswith("s_cbranch") or op == "s_branch":
            branches.append((len(instrs), args.strip()))
        elif re.match(r"(global|buffer|flat|scratch)_", op):
            # a load's first operand is its result, unless it goes to LDS
            reads = _sgprs(args if "store" in op or "lds" in op else args.partition(",")[2])
            if "lds" in op:
                reads.add("m0")
        elif op.startswith("v_"):
            writes = _sgprs(first)
            if re.search(r"_co_|div_scale|mad_[iu]64", op):  # a second, scalar result
                writes |= _sgprs(args.split(",")[1])
        instrs.append((op, writes, reads, states, number))
    for name, instrs, labels, branches in functions:
        before = [[i - 1] if i and not re.match(r"s_(branch|endpgm|setpc)", instrs[i - 1][0])
                  else [] for i in range(len(instrs))]
        for i, target in branches:
            if labels.get(target, len(instrs)) < len(instrs):
                before[labels[target]].append(i)
        yield name, instrs, before


def hazards(asm):
    """Vector memory reads of an SGPR too few wait states after a vector
    instruction's write of it, along every path."""
    found = []
    for name, instrs, before in _parse(asm):
        for i, (op, _, reads, _, number) in enumerate(instrs):
            paths = [(k, 0) for k in before[i]] if reads else []
            while paths:
                k, states = paths.pop()
                if instrs[k][1] & reads:
                    found.append(f"{name} line {number}: {op} {states} wait states after "
                                 f"{instrs[k][0]} in line {instrs[k][4]}")
                elif states + instrs[k][3] < WAIT_STATES:
                    paths += [(p, states + instrs[k][3]) for p in before[k]]
    return found


def test_the_scan_finds_a_pair_and_counts_its_wait_states():
    def kernel(*between):
        return "\n".join(["k:", "v_readfirstlane_b32 s5, v1", *between,
                          "global_load_lds_dwordx4 v0, s[4:5] offset:0", "s_endpgm"])
    assert len(hazards(kernel())) == 1
    assert len(hazards(kernel("s_nop 3"))) == 1
    assert hazards(kernel("s_nop 4")) == []
    assert hazards(kernel("s_nop 0", "v_mov_b32 v2, v3", "s_nop 2")) == []
    # along a branch: the write at the end of a loop, the read at its head
    loop = ["k:", "s_nop 4", ".L:", "global_load_lds_dwordx4 v0, s[4:5]",
            "v_readlane_b32 s4, v9, 3", "s_cbranch_scc1 .L", "s_endpgm"]
    assert len(hazards("\n".join(loop))) == 1
    loop.insert(5, "s_nop 4")
    assert hazards("\n".join(loop)) == []


def test_the_kernels_keep_the_wait_states(device_asm):
    assert len(device_asm) == 10, list(device_asm)  # five sources, two libraries
    assert sum(asm.count("global_load_lds") for asm in device_asm.values()) > 100
    found = {which: hazards(asm) for which, asm in device_asm.items() if hazards(asm)}
    assert not found, found


PROBE = """
#include "xattn_common.h"
using namespace xattn;
__global__ void probe(const char* a, int stride, float* out) {
    __shared__ __attribute__((aligned(16))) char lds[4096];
    const char* p = a + (size_t)(threadIdx.x >> 6) * stride;
    struct { DmaSrc a, b; } two;
    dma_base2(a, p, two.a, two.b);
    BODY
    wait_vmcnt<0>();
    lds_barrier();
    out[threadIdx.x] = ((float*)lds)[threadIdx.x];
}
"""


@pytest.mark.parametrize("dma", ["dma16_m0<0>", "dma16_untracked"])
def test_the_dma_takes_no_base_that_was_not_waited_for(tmp_path, dma):
    """The tightest code a kernel can write: refused with a plain pointer, and
    with the waiting base no pair in the assembly."""
    recipe = next(r for s, _, r in build_recipes() if "flash_f16" in s)

    def probe(name, base):
        source = tmp_path / f"{name}.hip"
        source.write_text(PROBE.replace(
            "BODY", f"{dma}({base}, 16u * (threadIdx.x & 63), lds_u32(lds));"))
        target = tmp_path / f"{name}.s"
        return assemble(str(source), recipe, target), target

    run, target = probe("plain", "uniform_ptr(p)")
    assert run.returncode != 0, "\n".join(hazards(target.read_text()))
    assert "DmaSrc" in run.stderr
    for name, base in (("one", "dma_base(p)"), ("two", "two.b")):
        run, target = probe(name, base)
        assert run.returncode == 0, run.stderr
        asm = target.read_text()
        assert "v_readfirstlane" in asm and "global_load_lds" in asm
        assert hazards(asm) == []
