"""The scheduled main loop of the Sage attention kernels as the compiler lays it
out: the device code is compiled to assembly (no GPU needed) and read."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "comfyui-turing-utils_amd", "csrc")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(head_dim, causal, split): [instructions of each basic block]}"""
    flags = re.search(r"^HIPFLAGS = ((?:.*\\\n)*.*)$", open(os.path.join(CSRC, "Makefile")).read(), re.M).group(1)
    out = tmp_path_factory.mktemp("asm") / "sage_attn.s"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), *flags.replace("\\\n", " ").split(), "--offload-device-only", "-S",
                    "sage_attn.hip", "-o", str(out)], cwd=CSRC, check=True, timeout=300)
    text = out.read_text()
    found = {}
    for m in re.finditer(r"^_ZN2tu12_GLOBAL__N_116sage_attn_kernelILi(\d+)ELb([01])ELb([01])E\S*:", text, re.M):
        body = text[m.end():text.index(".Lfunc_end", m.end())]
        blocks = []
        for b in re.split(r"^\.LBB[0-9_]+:", body, flags=re.M):
            blocks.append([ln.strip().split(";")[0] for ln in b.splitlines() if re.match(r"\t[a-z]", ln)])
        found[tuple(map(int, m.groups()))] = blocks
    assert len(found) == 8
    return found


FORMS = [(d, causal, split) for d in (64, 128) for causal in (0, 1) for split in (0, 1)]


@pytest.mark.parametrize("d,causal,split", FORMS)
def test_main_cluster_waits_for_single_fragments(kernels, d, causal, split):
    """The first MFMAs of a step need two of its first K fragments, not all:
    no wait for an empty LDS queue before them."""
    mfmas = 52 if d == 128 else 28
    clusters = [b for b in kernels[d, causal, split] if sum(i.startswith("v_mfma") for i in b) == mfmas and any("s_setprio" in i for i in b)]
    assert len(clusters) == 1
    block = clusters[0]
    first = next(i for i, x in enumerate(block) if x.startswith("v_mfma"))
    waits = [int(n) for x in block[:first] for n in re.findall(r"lgkmcnt\((\d+)\)", x)]
    reads = sum(x.startswith("ds_read") for x in block[:first])
    assert reads >= 4 and waits and min(waits) > 0, (reads, waits)


@pytest.mark.parametrize("causal,split", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_exponentials_of_head_dim_64_are_apart(kernels, causal, split):
    """At head_dim 64 a tile's exponentials alternate with other instructions
    (a run of eight holds the wave up)."""
    clusters = 0
    for block in kernels[64, causal, split]:
        runs = [len(r) for r in re.findall("E+", "".join("E" if x.startswith("v_exp") else "." for x in block))]
        if sum(runs) >= 16:
            clusters += 1
            assert sum(runs) <= 1.5 * len(runs) and max(runs) <= 3, runs
    assert clusters >= 2
