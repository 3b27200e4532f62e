"""Which branches the compiler takes for ones that lanes may decide differently in the kernels of the fused beam step.  A
barrier inside such a branch, or a loop that ends in one, leaves correct code to where the compiler puts its reloads of
spilled registers; every decision that a barrier depends on is the workgroup's, and has to look like that to the compiler."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "vectorlink-gpu_amd")
OPT = "/opt/rocm/llvm/bin/opt"

# a kernel of each kind: one iteration and several, without and with the sketch, with the bounds of all vectors, 16-byte loads and
# single elements, sums that become distances right away and together
KERNELS = """#include "beam_kernels.h"
namespace {
template __global__ void beam_step_kernel_w<2, 16, 4, 128, 8>(StepArgs);
template __global__ void beam_window_kernel<2, 16, 4, kRowAligned, 128, 6>(StepArgs);
template __global__ void beam_step_kernel<1, 64, 1, kRowScalar, 256>(StepArgs);
template __global__ void beam_window_kernel<1, 64, 4, kRowUnaligned, 256, 1>(StepArgs);
template __global__ void beam_window_kernel<2, 16, 2, kRowUnalignedSums, 128, 1>(StepArgs);
template __global__ void beam_window_kernel<1, 64, 8, kRowAligned, 256, 6>(StepArgs);
template __global__ void beam_step_sketch_kernel<3, 64, 1, 256, 3, 16, 1, 8>(StepArgs);
template __global__ void beam_window_sketch_kernel<3, 64, 1, 256, 3, 16, 1, 6>(StepArgs);
template __global__ void beam_window_near_kernel<3, 64, 2, 256, 3, 6>(StepArgs);
template __global__ void beam_window_near_kernel<8, 64, 1, 256, 4, 5>(StepArgs);
}
"""


def _flags():
    spec = importlib.util.spec_from_file_location("_vl_build", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    return build.FLAGS


def _kernels(text):
    """(name, blocks) of every function in what the uniformity printer says; a block: (successors, lanes may differ, barriers)"""
    for part in text.split("UniformityInfo for function '")[1:]:
        blocks = {}
        for body in part.split("\nBLOCK ")[1:]:
            (label, body) = body.split("\n", 1)
            (defs, terms) = body.split("END BLOCK")[0].split("TERMINATORS")
            blocks[label] = (re.findall(r"label %([\w.]+)", terms), "DIVERGENT" in terms, defs.count("s.barrier"))
        yield part.split("'")[0], blocks


def _barriers_behind_lanes(blocks):
    """Pairs (branch that lanes may take differently, block with a barrier before the lanes meet again)."""
    leave = "(exit)"
    succ = {b: (v[0] or [leave]) for b, v in blocks.items()}
    everything = set(succ) | {leave}
    after = {b: everything for b in succ}  # blocks that every path from b runs through
    after[leave] = {leave}
    moved = True
    while moved:
        moved = False
        for b in reversed(list(succ)):
            s = set.intersection(*[after[x] for x in succ[b]]) | {b}
            if s != after[b]:
                (after[b], moved) = (s, True)
    found = []
    for b, (_, lanes_differ, _) in blocks.items():
        meet = after[b] - {b}
        (seen, todo) = (set(), [x for x in succ[b] if x not in meet] if lanes_differ else [])
        while todo:
            x = todo.pop()
            if x in seen or x == leave:
                continue
            seen.add(x)
            todo += [y for y in succ[x] if y not in meet]
        found += [(b, x) for x in seen if blocks[x][2]]
    return found


@pytest.mark.skipif(shutil.which("hipcc") is None or not os.path.exists(OPT), reason="needs hipcc and LLVM's opt")
def test_no_barrier_of_the_step_lies_behind_a_branch_of_lanes(tmp_path):
    (src, ir) = (tmp_path / "kernels.hip", tmp_path / "kernels.ll")
    src.write_text(KERNELS)
    subprocess.run(["hipcc", "-x", "hip", *_flags(), "-I", os.path.join(PKG, "csrc"), "--cuda-device-only", "-S", "-emit-llvm",
                    str(src), "-o", str(ir)], check=True, capture_output=True)
    told = subprocess.run([OPT, "-disable-output", "-passes=print<uniformity>", str(ir)], check=True, capture_output=True, text=True)
    kernels = dict(_kernels(told.stderr))
    assert len(kernels) == 10 and all(sum(b[2] for b in k.values()) >= 8 for k in kernels.values())
    assert all(any(b[1] for b in k.values()) for k in kernels.values())  # (the printer does tell them apart)
    for name, blocks in kernels.items():
        assert not _barriers_behind_lanes(blocks), name
