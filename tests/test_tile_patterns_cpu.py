"""Tiles whose positions a map describes by a base and a pattern (tile_at / tile_rel of intra_maps.h and
intra_bwd_maps.h), compiled for the host: for every map, over ragged and ordinary shapes, each key or
column of such a tile has to sit where kpos / col_pos puts it.  The loaders of the kernels use the
pattern for whole tiles and the per-key position for the others."""
from test_key_rows_cpu import compile_and_run

SRC = r"""
#include <initializer_list>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include "intra_bwd_maps.h"
using namespace intra;

static long n_pattern = 0, n_other = 0, n_whole = 0;
static IntraGeom geom(int S) {
  IntraGeom ge;
  memset(&ge, 0, sizeof ge);
  ge.S = S; ge.G = 1; ge.window = 64; ge.width = 16; ge.text_len = 8; ge.pg = 1; ge.tm = 1; ge.blk = 64;
  ge.sink_chunk = 128;
  return ge;
}
template <class M, class P>
static void check(const M& m, int first, int n, P&& pos, const char* what) {
  for (int c = first; c < n; c += 64) {
    TileAt a;
    if (c + 64 <= n) ++n_whole;
    const bool cut = c + 64 > n, every = std::decay_t<M>::kEveryTile;
    if (every && !m.tile_at(c, a)) { printf("%s: tile %d follows no pattern\n", what, c); exit(1); }
    if ((cut && !every) || !m.tile_at(c, a)) { ++n_other; continue; }
    if (cut) ++n_other; else ++n_pattern;
    for (int i = 0; i < im_min(64, n - c); ++i)
      if (a.base + m.tile_rel(a.kind, i) != pos(c + i)) {
        printf("%s: tile %d, %d: %d, not %d\n", what, c, i, a.base + m.tile_rel(a.kind, i), pos(c + i));
        exit(1);
      }
  }
}
template <class MAP>
static void keys(IntraGeom ge, const char* what, int rows = 64) {
  geom_finish(ge);
  for (int set = 0; set < MAP::num_sets(ge); ++set)
    for (int t0 = 0; t0 < MAP(ge, set, 0).nq(); t0 += rows) {
      const MAP m(ge, set, t0);
      check(m, MAP::kHasPrefix ? 0 : m.klo(t0), m.nk(), [&](int t) { return m.kpos(t); }, what);
    }
}
template <class R>
static void columns(IntraGeom ge, const char* what) {
  geom_finish(ge);
  for (int set = 0; set < R::num_sets(ge); ++set)
    for (int r0 = 0; r0 < R::max_rows(ge); r0 += KEY_ROWS) {
      const R m(ge, set, r0);
      if (r0 >= m.n_rows()) continue;
      const int r1 = im_min(r0 + KEY_ROWS, m.n_rows()) - 1;
      check(m, m.block_lo(r0, r1), m.n_cols(), [&](int c) { return m.col_pos(c); }, what);
    }
}
static void report(const char* what, long& p, long& o) {
  printf("%s %ld %ld\n", what, n_pattern - p, n_other - o);
  p = n_pattern;
  o = n_other;
}

// every whole tile since the last call followed a pattern, and there was one
static void all_patterned(const char* what) {
  static long p = 0, w = 0;
  printf("%s %ld %ld\n", what, n_pattern - p, n_whole - w);
  p = n_pattern;
  w = n_whole;
}

static void aligned() {
  all_patterned("-");
  for (int S : {512, 4096}) {
    { IntraGeom ge = geom(S); ge.G = 2; keys<MapLlmScatter>(ge, "scatter"); all_patterned("scatter"); }
    { IntraGeom ge = geom(S); ge.G = 2; columns<KeyRowsOf<MapLlmScatter>>(ge, "scatter columns"); all_patterned("scatter_columns"); }
    { IntraGeom ge = geom(S); ge.G = 8; if (S >= 4096) { keys<MapLlmGather1>(ge, "gather1"); all_patterned("gather1"); } }
    { IntraGeom ge = geom(S); ge.G = 8; if (S >= 4096) { columns<KeyRowsOf<MapLlmGather1>>(ge, "gather1 columns"); all_patterned("gather1_columns"); } }
    { IntraGeom ge = geom(S); ge.window = 576; keys<MapLlmWindow>(ge, "window"); all_patterned("window"); }
    { IntraGeom ge = geom(S); ge.window = 576; columns<KeyRowsOf<MapLlmWindow>>(ge, "window columns"); all_patterned("window_columns"); }
    for (int ns : {0, 64}) {
      { IntraGeom ge = geom(S); ge.window = 575; ge.ns = ns; keys<MapLlmWindowSink>(ge, "window_sink"); all_patterned("window_sink"); }
      { IntraGeom ge = geom(S); ge.window = 575; ge.ns = ns; columns<KeyRowsWindowSink>(ge, "window_sink columns"); all_patterned("window_sink_columns"); }
      for (int off : {0, 1}) {
        IntraGeom ge = geom(S); ge.G = 2; ge.blk = 256; ge.off = off; ge.ns = ns;
        keys<MapLlmBlockScatter>(ge, "block_scatter"); all_patterned("block_scatter");
        columns<KeyRowsBlockScatter>(ge, "block_scatter columns"); all_patterned("block_scatter_columns");
      }
    }
    { IntraGeom ge = geom(S); ge.ns = 64; columns<KeyRowsFewSinks>(ge, "few sinks"); all_patterned("few_sinks"); }
    { IntraGeom ge = geom(S); ge.ns = 512; columns<KeyRowsText>(ge, "text"); all_patterned("text"); }
  }
  for (int width : {32, 64, 128}) {
    IntraGeom ge = geom(512 + width * width); ge.width = width; ge.text_len = 512;
    keys<MapImgScatter>(ge, "image scatter"); all_patterned("image_scatter");
    columns<KeyRowsImgGroup<false>>(ge, "grid keys"); all_patterned("grid_keys");
    columns<KeyRowsImgGroup<true>>(ge, "grid keys, text columns"); all_patterned("grid_keys_text_columns");
    columns<KeyRowsImgWindow>(ge, "window keys"); all_patterned("window_keys");
    for (int pg : {1, 2, 4}) { ge.pg = pg; keys<MapImgPatch>(ge, "patch runs"); all_patterned("patch_runs"); }
    for (int tm : {1, 2}) { ge.tm = tm; keys<MapImgTextRows>(ge, "text rows"); all_patterned("text_rows"); }
  }
}

int main(int argc, char**) {
  if (argc > 1) { aligned(); return 0; }
  long p = 0, o = 0;
  for (int S : {1, 63, 64, 65, 300, 777, 2048}) {
    for (int G : {1, 2, 3, 8, 13}) { IntraGeom ge = geom(S); ge.G = G; keys<MapLlmScatter>(ge, "scatter"); columns<KeyRowsOf<MapLlmScatter>>(ge, "scatter columns"); }
    for (int G : {2, 3, 8, 100}) { IntraGeom ge = geom(S); ge.G = G; keys<MapLlmGather1>(ge, "gather1"); columns<KeyRowsOf<MapLlmGather1>>(ge, "gather1 columns"); }
    for (int W : {64, 65, 130, 576}) { IntraGeom ge = geom(S); ge.window = W; keys<MapLlmWindow>(ge, "window"); columns<KeyRowsOf<MapLlmWindow>>(ge, "window columns"); }
    for (int W : {1, 63, 575}) for (int ns : {0, 1, 64, 700}) {
      IntraGeom ge = geom(S); ge.window = W; ge.ns = ns;
      keys<MapLlmWindowSink>(ge, "window_sink"); columns<KeyRowsWindowSink>(ge, "window_sink columns");
      if (ns) { columns<KeyRowsSinks>(ge, "sinks"); columns<KeyRowsText>(ge, "text"); }
      if (ns && ns <= 64) columns<KeyRowsFewSinks>(ge, "few sinks");
    }
    for (int G : {1, 2, 3}) for (int off = 0; off < G; ++off) for (int ns : {0, 1, 64}) {
      IntraGeom ge = geom(S); ge.G = G; ge.blk = off != 0 ? 256 : 64; ge.off = off; ge.ns = ns;
      keys<MapLlmBlockScatter>(ge, "block_scatter"); columns<KeyRowsBlockScatter>(ge, "block_scatter columns");
    }
  }
  report("llm", p, o);
  for (int width : {16, 24, 32, 40, 64, 128}) for (int text : {8, 72, 128, 512}) {
    IntraGeom ge = geom(text + width * width); ge.width = width; ge.text_len = text;
    keys<MapImgScatter>(ge, "image scatter"); columns<KeyRowsImgGroup<false>>(ge, "grid keys"); columns<KeyRowsImgGroup<true>>(ge, "grid keys, text columns");
    columns<KeyRowsImgWindow>(ge, "window keys");
    for (int pg : {1, 2, 4}) { if ((width / 8) % pg) continue; ge.pg = pg; keys<MapImgPatch>(ge, "patch runs"); }
    for (int tm : {1, 2}) { ge.tm = tm; keys<MapImgTextRows>(ge, "text rows"); }
  }
  report("image", p, o);
  return 0;
}
"""


def test_patterned_tiles_sit_where_the_maps_put_their_keys(tmp_path):
    out = [line.split() for line in compile_and_run(tmp_path, SRC).splitlines()]
    assert [line[0] for line in out] == ["llm", "image"], out
    for kind, pattern, other in out:  # both kinds of tiles occur
        assert int(pattern) > 1000 and int(other) > 100, (kind, pattern, other)


def test_every_whole_tile_of_aligned_shapes_follows_a_pattern(tmp_path):
    """Map by map: one that answers false there would leave its loader with positions row by row, unnoticed."""
    lines = [line.split() for line in compile_and_run(tmp_path, SRC, args=["aligned"]).splitlines()][1:]
    assert len({what for what, _, _ in lines}) == 18, lines
    for what, pattern, whole in lines:
        assert int(pattern) == int(whole) > 0, (what, pattern, whole)
