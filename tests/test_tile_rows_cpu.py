"""Block Scatter's forward loader: which tiles of 64 keys it requests by one position (tile_rows), compiled for the
host.  Every tile that lies inside a part of the key list is one, none else, and its keys are where kpos says."""
import pytest

from test_key_rows_cpu import compile_and_run

SRC = r"""
#include <stdio.h>
#include "intra_maps.h"

int main() {  // every line of the input: S G blk off ns pos
  int S, G, blk, off, ns, pos;
  while (scanf("%d %d %d %d %d %d", &S, &G, &blk, &off, &ns, &pos) == 6) {
    IntraGeom ge{};
    ge.S = S; ge.G = G; ge.blk = blk; ge.off = off; ge.ns = ns;
    ge.width = 64; ge.text_len = 64; ge.pg = ge.tm = 1;
    geom_finish(ge);
    int full = 0, by_rows = 0, wrong = 0, straight = 0;
    for (int set = 0; set < MapLlmBlockScatter::num_sets(ge); ++set)
      for (int t0 = 0; t0 < MapLlmBlockScatter(ge, set, 0).nq(); t0 += pos) {
        const MapLlmBlockScatter map(ge, set, t0);
        for (int t = 0; t < map.nk(); t += 64) {
          const bool whole = t + 64 <= map.nk();
          bool run = whole;
          for (int i = 1; run && i < 64; ++i) run = map.kpos(t + i) == map.kpos(t) + i;
          TileRows tr;
          const bool rows = map_tile_rows(map, t, tr);
          full += whole;
          straight += run;
          by_rows += rows;
          wrong += rows != run;
          for (int i = 0; rows && i < 64; ++i) wrong += tr.base + i / 4 * tr.group_step + i % 4 * tr.row_step != map.kpos(t + i);
        }
      }
    printf("%d %d %d %d\n", full, straight, by_rows, wrong);
  }
  return 0;
}
"""

CASES = [(S, G, blk, off, ns, pos) for S in (1, 63, 64, 300, 1000, 4100) for G, off in ((1, 0), (2, 0), (2, 1), (8, 3))
         for blk in (64, 256) for ns in (0, 4, 64) for pos in (32, 64, 128) if off == 0 or blk % pos == 0]


def test_tiles_inside_a_part_of_the_list(tmp_path):
    out = compile_and_run(tmp_path, SRC, "\n".join(" ".join(map(str, c)) for c in CASES) + "\n")
    lines = [tuple(map(int, line.split())) for line in out.splitlines()]
    assert len(lines) == len(CASES)
    for case, (full, straight, by_rows, wrong) in zip(CASES, lines):
        assert wrong == 0 and by_rows == straight, (case, full, straight, by_rows, wrong)
        if case[4] % 64 == 0:  # no tile straddles the sinks' end
            assert by_rows == full, (case, full, by_rows)
    assert sum(by_rows for _, _, by_rows, _ in lines) > 10000
