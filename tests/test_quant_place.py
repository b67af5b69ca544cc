"""Where a batch's quantised rows lie (chunk_place, quant_formats.h): the
function k_quant_rows takes its row, chunk and row offset from, compiled for
the host and checked against Python's integers up to the largest batches the
grouped calls accept (rows of up to 4 GiB, 2^24 pairs)."""
from __future__ import annotations

import os
import random
import shutil
import subprocess

import pytest

from helpers import ROOT

CSRC = os.path.join(ROOT, "sabah-moe-accelerator_amd", "csrc")
MAIN = r"""
#include <cstdio>
#include "quant_formats.h"
int main() {
    int q, nch, stride;
    while (std::scanf("%d %d %d", &q, &nch, &stride) == 3) {
        const sabah::ChunkPlace p = sabah::chunk_place(q, nch, stride);
        std::printf("%d %d %zu\n", p.row, p.chunk, p.offset);
    }
}
"""


def test_rows_past_2_gib_and_past_2_million_chunks(tmp_path):
    cxx = shutil.which("g++")
    if not cxx or not os.path.isdir("/opt/rocm/include/hip"):
        pytest.skip("no host compiler or HIP headers")
    src, exe = tmp_path / "place.cpp", tmp_path / "place"
    src.write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + CSRC, str(src), "-o",
                    str(exe)], check=True, capture_output=True)
    rng = random.Random(7)
    # (chunks per row, row stride, rows): the last rows of batches up to the limits
    batches = [(16, 4864, 450_000), (56, 17248, 124_508), (128, 38912, 65_536), (3, 912, (1 << 32) // 912),
               (8, 2464, 1 << 24), (1, 304, (1 << 32) // 304)]
    cases = []
    for nch, stride, rows in batches:
        for r in [0, 1, rows // 2, rows - 1] + [rng.randrange(rows) for _ in range(2000)]:
            for c in {0, nch - 1, rng.randrange(nch)}:
                cases.append((r, c, nch, stride))
    text = "".join("%d %d %d\n" % (r * nch + c, nch, stride) for r, c, nch, stride in cases)
    out = subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout.splitlines()
    assert len(out) == len(cases)
    for (r, c, nch, stride), line in zip(cases, out):
        assert tuple(map(int, line.split())) == (r, c, r * stride), (r, c, nch, stride)
