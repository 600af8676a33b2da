"""The key-row maps of the dK / dV launch (intra_amd/csrc/intra_bwd_maps.h), compiled for the host: how
the queries of the leading keys (LLM sinks, image text keys) are cut into chunks, the columns of block
Scatter's row blocks, and what the maps call their longest row block."""
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
    printf("%d %d %lld\n", chunk, (S + chunk - 1) / chunk, (long long)leading_floats(S, B, Hkv, ns));
  }
  return 0;
}
"""


def compile_and_run(tmp_path, source, text="", args=()):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(source)
    subprocess.run([gxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "intra_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe), *args], input=text, check=True, capture_output=True, text=True).stdout


def splits(tmp_path, shapes):
    """(queries of a chunk, chunks, floats of room for partial sums) of every (S, B, Hkv, ns, cus)"""
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
        assert n == 1 or 2 * n * B * Hkv * ns * 128 <= room, what


def test_the_gpu_tests_meet_every_kind_of_split(tmp_path):
    from test_backward_gpu import SINK_CHUNKS
    counts = {n for _, n, _ in splits(tmp_path, [(S, B, Hkv, ns, 256) for B, S, _, Hkv, ns in SINK_CHUNKS])}
    assert 1 in counts and any(1 < n < 8 for n in counts) and any(n > 8 and n % 8 for n in counts), counts


def test_workspace_is_what_the_finest_split_writes(tmp_path, lib):
    """No room that no launch uses: nothing for a single chunk, both results of the chunks otherwise."""
    for S, B, Hkv, width in ((4608, 1, 3, 64), (4608, 1, 24, 64), (4608, 2, 24, 64), (16896, 1, 16, 128), (16896, 2, 24, 128)):
        (_, n, _), = splits(tmp_path, [(S, B, Hkv, 512, 1 << 20)])
        want = 2 * B * S * Hkv + (2 * n * B * Hkv * 512 * 128 if n > 1 else 0)
        assert lib.intra_image_bwd_workspace(B, S, Hkv, Hkv, 0, width, 512) == want, (S, B, Hkv)
    for S, B, Hkv, ns in ((64, 1, 1, 4), (390, 1, 2, 130), (1000, 3, 28, 64), (6000, 1, 8, 64), (320, 2, 82, 3)):
        (_, n, _), = splits(tmp_path, [(S, B, Hkv, ns, 1 << 20)])
        want = 2 * B * S * Hkv + (2 * n * B * Hkv * ns * 128 if n > 1 else 0)
        assert lib.intra_llm_bwd_workspace(B, S, Hkv, Hkv, 9, 2, 575, 256, 0, ns) == want, (S, B, Hkv, ns)


COLS = r"""
#include <stdio.h>
#include <string.h>
#include "intra_bwd_maps.h"
using namespace intra;

int main() {  // every line of the input: S G block offset; output: key block, then the positions of its columns
  int S, G, blk, off;
  while (scanf("%d %d %d %d", &S, &G, &blk, &off) == 4) {
    IntraGeom ge;
    memset(&ge, 0, sizeof ge);
    ge.S = S; ge.G = G; ge.window = 64; ge.width = 16; ge.text_len = 8; ge.pg = 1; ge.tm = 1; ge.blk = blk; ge.off = off;
    ge.sink_chunk = 1024;
    geom_finish(ge);
    for (int set = 0; set < G; ++set)
      for (int r0 = 0; r0 < KeyRowsBlockScatter::max_rows(ge); r0 += KEY_ROWS) {
        const KeyRowsBlockScatter m(ge, set, r0);
        if (r0 >= m.n_rows()) continue;
        const int r1 = (r0 + KEY_ROWS < m.n_rows() ? r0 + KEY_ROWS : m.n_rows()) - 1;
        printf("%d", m.row_pos(r0));
        const int cb = m.block_lo(r0, r1);
        for (int c = cb; c <= m.block_hi(r0, r1); ++c) {
          printf(" %d", m.col_pos(c));
          if (m.col_pos(c) - c != m.tile_shift(cb + ((c - cb) & ~63))) printf(" not the tile's shift");
        }
        printf("\n");
      }
    printf("end\n");
  }
  return 0;
}
"""


@pytest.mark.parametrize("S,G,blk,off", [
    (1, 1, 256, 0), (255, 2, 256, 1), (256, 2, 256, 1), (257, 2, 256, 1), (1000, 3, 256, 2), (1000, 3, 64, 0),
    (1100, 4, 256, 1), (1537, 2, 512, 1), (1537, 2, 512, 0), (2048, 8, 256, 7), (700, 64, 256, 63), (900, 1, 320, 0)])
def test_columns_of_block_scatter_row_blocks(tmp_path, S, G, blk, off):
    """From the first key of a row block on: the later queries of its block and the blocks that see it, in order."""
    out = compile_and_run(tmp_path, COLS, f"{S} {G} {blk} {off}\n").splitlines()
    assert out[-1] == "end" and len(out) > 1
    for line in out[:-1]:
        first, *cols = map(int, line.split())
        kb = first // blk
        own = [p for p in range(first, min(S, (kb + 1) * blk))]
        seen_by = [qb for qb in range(kb + 1, -(-S // blk)) if (qb + off) % G == kb % G]
        assert cols == own + [p for qb in seen_by for p in range(qb * blk, min(S, (qb + 1) * blk))], (S, G, blk, off, first)


LONGEST = r"""
#include <stdio.h>
#include <string.h>
#include <initializer_list>
#include "intra_bwd_maps.h"
using namespace intra;

template <class R>
static void check(const char* name, IntraGeom ge) {
  geom_finish(ge);
  int most = 0;
  for (int set = 0; set < R::num_sets(ge); ++set)
    for (int r0 = 0; r0 < R::max_rows(ge); r0 += KEY_ROWS) {
      const R m(ge, set, r0);
      if (r0 >= m.n_rows()) continue;
      const int r1 = im_min(r0 + KEY_ROWS, m.n_rows()) - 1;
      most = im_max(most, m.block_hi(r0, r1) - m.block_lo(r0, r1) + 1);
    }
  if (most != R::longest(ge)) printf("%s: S %d G %d block %d offset %d window %d width %d: %d columns, longest() says %d\n", name,
                                     ge.S, ge.G, ge.blk, ge.off, ge.window, ge.width, most, R::longest(ge));
}

int main() {
  IntraGeom ge0;
  memset(&ge0, 0, sizeof ge0);
  ge0.G = 1; ge0.window = 64; ge0.width = 16; ge0.text_len = 8; ge0.pg = 1; ge0.tm = 1; ge0.blk = 256; ge0.sink_chunk = 1024;
  for (int S : {1, 100, 256, 300, 1000, 4096, 6000}) {
    for (int G : {1, 2, 3, 8}) for (int off = 0; off < G; ++off) { IntraGeom ge = ge0; ge.S = S; ge.G = G; ge.off = off; check<KeyRowsBlockScatter>("block scatter", ge); }
    for (int w : {1, 255, 575, 5000}) { IntraGeom ge = ge0; ge.S = S; ge.window = w; check<KeyRowsWindowSink>("window", ge); }
  }
  for (int width = 16; width <= 192; width += 8) for (int text : {8, 512}) {
    IntraGeom ge = ge0;
    ge.S = text + width * width; ge.width = width; ge.text_len = text;
    check<KeyRowsImgWindow>("image gather 0", ge);
    check<KeyRowsImgGroup<false>>("image scatter", ge);
  }
  return 0;
}
"""


def test_longest_row_block(tmp_path):
    """Which workgroups of the dK / dV launch come first is decided by it."""
    assert compile_and_run(tmp_path, LONGEST) == ""
