"""How the queries of the leading keys (LLM sinks, image text keys) are cut into chunks for the dK / dV
launch, and what the launch's row maps (intra_amd/csrc/intra_bwd_maps.h) say about their row blocks,
compiled for the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <stdio.h>
#include <string.h>
#include "intra_bwd_maps.h"
using namespace intra;

int main() {  // every line of the input: S B Hkv ns cus
  int S, B, Hkv, ns, cus;
  while (scanf("%d %d %d %d %d", &S, &B, &Hkv, &ns, &cus) == 5) {
    const int chunk = leading_chunk(S, B, Hkv, ns, cus);
    printf("%d %d %d\n", chunk, (S + chunk - 1) / chunk, workspace_chunks(S, B, Hkv, ns));
  }
  return 0;
}
"""


def compile_and_run(tmp_path, source, text=""):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(source)
    subprocess.run([gxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "intra_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout


def splits(tmp_path, shapes):
    """(queries of a chunk, chunks, chunks of one result that the workspace holds) of every (S, B, Hkv, ns, cus)"""
    out = compile_and_run(tmp_path, SRC, "\n".join(" ".join(map(str, s)) for s in shapes) + "\n")
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_no_more_workgroups_on_leading_keys_than_cus(tmp_path):
    """One round at most, unless a single chunk already has more; both results fit the workspace; chunks of a
    multiple of 64 queries that cover the sequence."""
    shapes = [(S, B, Hkv, ns, cus) for S in (1, 64, 130, 700, 4608, 6000, 16896, 65536)
              for B, Hkv in ((1, 1), (1, 3), (2, 6), (1, 8), (1, 12), (2, 8), (1, 24), (1, 32), (2, 24), (3, 82))
              for ns in (1, 64, 65, 128, 129, 200, 256, 512) for cus in (64, 256, 304, 320, 400)]
    for (S, B, Hkv, ns, cus), (chunk, n, room) in zip(shapes, splits(tmp_path, shapes)):
        what = f"S={S} B={B} Hkv={Hkv} ns={ns} cus={cus}: {n} chunks of {chunk}"
        assert chunk % 64 == 0 and (n - 1) * chunk < S <= n * chunk, what
        assert n == 1 or n * B * Hkv * -(-ns // 128) <= cus, what
        assert n == 1 or 2 * n <= room, what
