"""The kernels whose waves hand values from lane to lane through LDS without a barrier rely on the order of one wave's LDS
accesses.  The hardware keeps it; the compiler only has to where a fence stands, because what another lane wrote is
nothing that it can see.  Compiled here to LLVM IR with the library's own flags, no GPU needed."""
import os
import re
import shutil
import subprocess

import pytest

from openagents_amd import build

ACCESS = re.compile(r"^\s+(?:%\S+ = (load)\b|(store)\b).*ptr addrspace\(3\)")


def unordered(ir):
    """(function, instruction) of every LDS load that a store can reach without a fence between them, and of every store that
    a load can reach: a fixpoint over the blocks of each function."""
    found, kernels = [], 0
    for name, body in re.findall(r"^define [^\n]*amdgpu_kernel[^\n]* @(\w+)\([^\n]*\{\n(.*?)^\}", ir, re.S | re.M):
        kernels += 1
        blocks, succ, label = {"entry": []}, {}, "entry"
        for line in body.split("\n"):
            m = re.match(r"^(\S+):", line)
            if m:
                label = m.group(1)
                blocks[label] = []
            else:
                blocks[label].append(line)
        for label, lines in blocks.items():
            succ[label] = re.findall(r"label %([\w.]+)", "\n".join(lines))
        state, todo = {label: frozenset() for label in blocks}, list(blocks)
        bad = set()
        while todo:
            label = todo.pop()
            pending = set(state[label])
            for line in blocks[label]:
                if re.match(r"^\s+fence ", line):
                    pending.clear()
                m = ACCESS.match(line)
                if m:
                    kind = m.group(1) or m.group(2)
                    if pending - {kind}:
                        bad.add(line.strip())
                    pending.add(kind)
            for to in succ[label]:
                if not pending <= state[to]:
                    state[to] = state[to] | pending
                    todo.append(to)
        found += [(name, line) for line in sorted(bad)]
    return kernels, found


@pytest.mark.parametrize("stem", ["psn_mvb", "psn_th_q4_0", "psn_th_q8_0", "psn_th_q4_K", "psn_th_q5_K", "psn_th_q6_K"])
def test_lane_to_lane_hand_over_is_fenced(stem, tmp_path):
    hipcc = build._hipcc()
    if not shutil.which(hipcc):
        pytest.skip("no hipcc")
    (src, defs), = [(src, defs) for s, src, defs in build.CODE_OBJECTS if s == stem]
    out = tmp_path / "k.ll"
    flags = [f for f in build.DEVICE_FLAGS if f != "--genco"]
    subprocess.run([hipcc, *flags, *defs, "-I", build.CSRC, "--cuda-device-only", "-S", "-emit-llvm", "-o", str(out), os.path.join(build.CSRC, src)],
                   check=True, capture_output=True)
    kernels, found = unordered(out.read_text())
    assert kernels >= 2
    assert not found, (len(found), found[:4])
