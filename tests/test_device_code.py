"""The compiled wave engine: what its kernels keep in scratch memory, and where they store it.

The untraced kernels for indexes below 2^32 symbols hold the state of a round in registers: what they spill
is a thread's constants, stored once in straight-line code before their loops, with every lane on. Builds
of the same source that stored spilled values from several branches of the loops gave wrong records."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from galn_amd import build


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "search.s")
    r = subprocess.run([build.HIPCC, *build.HIP_FLAGS, f"-I{build.INC}", "--cuda-device-only", "-S", "-o", out,
                        os.path.join(build.CSRC, "galn_search.hip")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    found, name = {}, None
    with open(out) as f:
        for line in f:
            m = re.match(r"^(_ZN\S*7k_heavyILb(\d)ELb(\d)ELi(\d)\S*):", line)
            if m:
                name = (int(m.group(2)), int(m.group(3)), int(m.group(4)))  # traced, 2^32 symbols, waves
                found[name] = []
            elif line.startswith(".Lfunc_end"):
                name = None
            elif name:
                found[name].append(line)
    return found


@pytest.mark.parametrize("waves", [1, 4])
def test_spilled_values_are_stored_before_the_loops(waves, kernels):
    assert len(kernels) == 8
    block, blocks, on, loop = "entry", [], True, False
    for line in kernels[0, 0, waves]:
        if line.startswith(".LBB"):
            block, on, loop = line.split(":")[0], True, "Loop" in line
        code = line.split(";")[0]
        if re.search(r"\bexec\b", code):
            on = False  # lanes may be off from here to the end of the block
        if "scratch_store" in code:
            blocks.append(block)
            assert on and not loop, line
    assert len(set(blocks)) <= 1, blocks


@pytest.mark.parametrize("which", [(t, w, n) for t in (0, 1) for w in (0, 1) for n in (1, 4)])
def test_the_register_of_spilled_scalars_holds_nothing_else(which, kernels):
    lines = [ln.split(";")[0].strip() for ln in kernels[which]]
    lanes = {m.group(1) for ln in lines if (m := re.match(r"v_writelane_b32 v(\d+),", ln))}
    for ln in lines:
        if ln.startswith(("v_writelane", "v_readlane")):
            continue
        used = {n for n in re.findall(r"\bv(\d+)\b", ln)}
        used |= {str(k) for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", ln) for k in range(int(a), int(b) + 1)}
        assert not used & lanes, ln
