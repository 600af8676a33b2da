// Row maps of the backward kernels: which "columns" a block of "rows" meets.
//
// dQ: rows are the queries of a set and columns its keys - the forward index map as it is
// (QueryRows).  dK / dV: rows are keys and columns the queries that see them.  For the patterns
// whose sets number queries and keys alike, the query range of a key starts at the key and ends
// where the forward map says (KeyRowsOf).  Block Scatter with a stripe offset and the
// per-token window have their own inverse maps.  Keys that are sinks are seen by every later
// query of every set; they are left out of those maps' results (`store`) and get row blocks of
// their own in the same launch (KeyRowsSinks), split over chunks of queries whose partial sums a
// small kernel adds up.
//
// Interface (host and device):
//   static num_sets(ge), max_rows(ge)      grid size: sets per (batch, kv head), rows of the largest
//   RowMap(ge, set, r0)                    r0: first row of the row block (rows r0 .. r0+255 at most, keys r0 .. r0+127)
//   n_rows(), n_cols()
//   row_pos(t), col_pos(c)                 token positions
//   lo(t), hi(t)                           row t meets the columns lo..hi (and those below kpre())
//   block_lo(r0, r1), block_hi(r0, r1)     union of the ranges of rows r0..r1
//   store(pos)                             whether the result row of token pos is written here
//   kBlockPredicate / sees(t, c)           maps whose rows do not meet one range of columns say per
//                                          row and 32-column block (first column c) whether the row
//                                          meets the block - all of it or nothing
//   tile_at(c, a), tile_rel(kind, i)       where the 64 columns from c on sit (TileAt in intra_maps.h), asked
//                                          for tiles of 64 from block_lo on that lie inside the column list
//   kEveryTile                             tile_at is true for each of them, and for one cut by the end of the list
//   kAccumulate                            the results are added to rows another pass has written
//   static longest(ge)                     columns of the longest row block (maps that share a launch with leading keys)
//   alternates<RowMap>                     rows 0..63 and 64..127 are the same keys twice over: the
//                                          first meet the even blocks of 32 columns, the second the odd
//                                          ones, and the results of the two are added
#pragma once
#include "intra_maps.h"

namespace intra {

constexpr int KEY_ROWS = 128;  // keys of a row block of the dK / dV launch

template <class RMAP>
constexpr bool alternates = false;

template <class MAP>
struct QueryRows {
  MAP m;
  static IM_HD int num_sets(const IntraGeom& ge) { return MAP::num_sets(ge); }
  static IM_HD int max_rows(const IntraGeom& ge) { return MAP::max_nq(ge); }
  IM_HD QueryRows(const IntraGeom& ge, int set, int r0) : m(ge, set, r0) {}
  IM_HD int n_rows() const { return m.nq(); }
  IM_HD int n_cols() const { return m.nk(); }
  IM_HD int kpre() const { return m.kpre(); }
  IM_HD int row_pos(int t) const { return m.qpos(t); }
  IM_HD int col_pos(int c) const { return m.kpos(c); }
  IM_HD bool tile_at(int c, TileAt& a) const { return m.tile_at(c, a); }
  IM_HD int tile_rel(int kind, int i) const { return m.tile_rel(kind, i); }
  IM_HD int lo(int t) const { return m.klo(t); }
  IM_HD int hi(int t) const { return im_min(m.khi(t), m.nk() - 1); }
  IM_HD int block_lo(int r0, int) const { return m.kpre() > 0 ? 0 : m.klo(r0); }
  IM_HD int block_hi(int, int r1) const { return hi(r1); }
  IM_HD bool store(int) const { return true; }
  static constexpr bool kEveryTile = MAP::kEveryTile;
  static constexpr bool kBlockPredicate = false, kAccumulate = false;
  IM_HD bool sees(int, int) const { return true; }
};

// Keys of a set whose queries and keys carry the same numbering and whose queries see keys up to
// their own (LLM Scatter, Gather 1, window): key r is seen by the queries from r to the last one
// whose lower key bound does not exceed r (last_query).  In closed form: a search for the two ends
// in the forward map's bounds was six chains of a dozen dependent iterations in front of the first
// request of every workgroup.
template <class MAP>
struct KeyRowsOf {
  MAP m;
  static IM_HD int num_sets(const IntraGeom& ge) { return MAP::num_sets(ge); }
  static IM_HD int max_rows(const IntraGeom& ge) { return MAP::max_nq(ge); }
  IM_HD KeyRowsOf(const IntraGeom& ge, int set, int) : m(ge, set, 0) {}
  IM_HD int n_rows() const { return m.nk(); }
  IM_HD int n_cols() const { return m.nq(); }
  IM_HD int kpre() const { return 0; }
  IM_HD int row_pos(int t) const { return m.kpos(t); }
  IM_HD int col_pos(int c) const { return m.qpos(c); }
  IM_HD bool tile_at(int c, TileAt& a) const { return m.tile_at(c, a); }
  IM_HD int tile_rel(int kind, int i) const { return m.tile_rel(kind, i); }
  IM_HD int lo(int r) const { return r; }
  IM_HD int hi(int r) const { return im_min(m.last_query(r), m.nq() - 1); }
  IM_HD int block_lo(int r0, int) const { return lo(r0); }
  IM_HD int block_hi(int, int r1) const { return hi(r1); }
  IM_HD bool store(int) const { return true; }
  static constexpr bool kEveryTile = MAP::kEveryTile;
  static constexpr bool kBlockPredicate = false, kAccumulate = false;
  IM_HD bool sees(int, int) const { return true; }
};

// Keys of group gk of block Scatter (blocks kb = gk mod G), any stripe offset.  Without offset the
// queries that see them are the later tokens of the same group.  With offset `off` a key of block
// kb is seen by the later queries of its own block and by all queries of the blocks kb + G - off,
// kb + 2G - off, ... (the query blocks qb > kb with (qb + off) mod G = gk); the columns of a row
// block are numbered [own block][those blocks], which needs the row block inside one key block
// (block size a multiple of 256).  Sinks (positions < n_sink) are not stored here.
struct KeyRowsBlockScatter {
  int G, blk, gk, off, n, skip, a, own, ncols;
  uint32_t own_pos, far_pos, far_step;  // position minus column: in the own block, in the first one behind it; more per further block
  FastDiv dBlk;
  static IM_HD int num_sets(const IntraGeom& ge) { return ge.G; }
  static IM_HD int max_rows(const IntraGeom& ge) { return MapLlmBlockScatter::max_nq(ge); }
  IM_HD KeyRowsBlockScatter(const IntraGeom& ge, int set, int r0) {
    G = ge.G;
    blk = ge.blk;
    off = ge.off;
    dBlk = ge.dBlk;
    gk = set;
    skip = im_min(ge.ns, ge.S);
    n = MapLlmBlockScatter::group_size(ge, gk);
    a = (int)fd_div(r0, dBlk);
    far_step = (uint32_t)(G - 1) * (uint32_t)blk;
    if (off == 0) {
      own = 0;
      own_pos = 0;
      far_pos = (uint32_t)gk * (uint32_t)blk;
      ncols = n;
    } else {
      const int S = ge.S, kb = a * G + gk, qb0 = kb + G - off;
      const int nbt = (int)fd_div(S + blk - 1, dBlk);  // blocks in the sequence, the last one maybe short
      int later = 0;
      if (qb0 < nbt) {
        const int cnt = (int)fd_div(nbt - 1 - qb0, ge.dG) + 1;  // blocks qb0, qb0 + G, ... below nbt
        const int last = qb0 + (cnt - 1) * G;
        later = (cnt - 1) * blk + im_min(blk, S - last * blk);
      }
      own = im_max(0, im_min(blk, S - kb * blk));
      own_pos = (uint32_t)kb * (uint32_t)blk;
      far_pos = (uint32_t)qb0 * (uint32_t)blk - (uint32_t)own;
      ncols = own + later;
    }
  }
  IM_HD int n_rows() const { return n; }
  IM_HD int n_cols() const { return ncols; }
  IM_HD int kpre() const { return 0; }
  IM_HD int row_pos(int t) const {
    const int b = (int)fd_div(t, dBlk);
    return (b * G + gk) * blk + (t - b * blk);
  }
  // Blocks start at multiples of 64 columns, so a tile lies inside one.  Worked out once per tile, in
  // scalars: per lane and group of rows it was a chain of branches on `off` and on the own block, whose
  // scalars were spilled and read back in the main loop of the launch that more than 64 sinks share
  // (19 lane reads and 36 branches per step there, 27 branches elsewhere).  Training steps,
  // G = 2, S = 8192: offset 1 and 128 sinks at 32 / 32 heads 1432 -> 1334 us, 64 sinks at 32 / 8 heads
  // 1248 -> 1217, neither offset nor sinks 1121 -> 1107.
  IM_HD int tile_shift(int c) const {
    return (int)(c < own ? own_pos : far_pos + fd_div((uint32_t)(c - own), dBlk) * far_step);
  }
  IM_HD int col_pos(int c) const { return c + tile_shift(c); }
  IM_HD bool tile_at(int c, TileAt& a) const {
    a = TileAt{c + tile_shift(c), TILE_LINEAR};
    return true;
  }
  IM_HD int tile_rel(int, int i) const { return i; }
  static int longest(const IntraGeom& ge) { return KeyRowsBlockScatter(ge, 0, 0).n_cols(); }  // (the first block's)
  IM_HD int lo(int t) const { return off == 0 ? t : t - a * blk; }
  IM_HD int hi(int) const { return ncols - 1; }
  IM_HD int block_lo(int r0, int) const { return lo(r0); }
  IM_HD int block_hi(int, int) const { return ncols - 1; }
  IM_HD bool store(int pos) const { return pos >= skip; }
  static constexpr bool kEveryTile = true;
  static constexpr bool kBlockPredicate = false, kAccumulate = false;
  IM_HD bool sees(int, int) const { return true; }
};

// Keys of the per-token window with sinks: key j is seen by the queries j .. j + window - 1.
// Sinks (j < n_sink; seen by every later query) are not stored here.
struct KeyRowsWindowSink {
  int S, window, skip;
  static IM_HD int num_sets(const IntraGeom&) { return 1; }
  static IM_HD int max_rows(const IntraGeom& ge) { return ge.S; }
  static int longest(const IntraGeom& ge) { return (int)im_min64((int64_t)ge.window + KEY_ROWS - 1, ge.S); }
  IM_HD KeyRowsWindowSink(const IntraGeom& ge, int, int) {
    S = ge.S;
    window = ge.window;
    skip = im_min(ge.ns, ge.S);
  }
  IM_HD int n_rows() const { return S; }
  IM_HD int n_cols() const { return S; }
  IM_HD int kpre() const { return 0; }
  IM_HD int row_pos(int t) const { return t; }
  IM_HD int col_pos(int c) const { return c; }
  IM_HD bool tile_at(int c, TileAt& a) const {
    a = TileAt{c, TILE_LINEAR};
    return true;
  }
  IM_HD int tile_rel(int, int i) const { return i; }
  IM_HD int lo(int t) const { return t; }
  IM_HD int hi(int t) const { return (int)im_min64((int64_t)t + window - 1, S - 1); }
  IM_HD int block_lo(int r0, int) const { return r0; }
  IM_HD int block_hi(int, int r1) const { return hi(r1); }
  IM_HD bool store(int pos) const { return pos >= skip; }
  static constexpr bool kEveryTile = true;
  static constexpr bool kBlockPredicate = false, kAccumulate = false;
  IM_HD bool sees(int, int) const { return true; }
};

// Chunks of queries that the row blocks of the `ns` leading keys (LLM sinks, image text keys) are cut
// into, and their length, a multiple of 64 and at least 128 (except for the last).  Half as many as
// would give every CU of a device of WS_CUS CUs one block of 256 keys, so that the fp32 partial sums of
// dk and dv are as many as one such block per CU would have of one result, and their room
// (leading_floats) does not depend on the device.  Nor are there more workgroups on leading keys than the
// device has CUs: a few too many are a second round of the longest kind on a few CUs, which everything
// else waits for.  With 288 - 320 workgroups on 256 CUs against 192 - 256 (training steps, us): image
// Scatter 2048^2 at 12 heads 1211 -> 1164, at 6 heads 691 -> 657; Gather 0 at 24 heads 384 -> 361
// (1024^2) and 1234 -> 1174 (2048^2); 256 sinks, 32 / 8 heads, S = 16384: window 575 1202 -> 1124,
// block Scatter 4750 -> 4660.  (Slower: 1000 sinks at S = 3000, 336 -> 348, where 5 short chunks
// behind the window's row blocks fill the rounds better than 4.)
constexpr int WS_CUS = 320;
inline int chunk_length(int S, int64_t chunks) {
  if (chunks < 1) chunks = 1;
  return (int)(64 * ((S + 64 * chunks - 1) / (64 * chunks)));
}
inline int chunk_count(int S, int chunk) { return (S + chunk - 1) / chunk; }
inline int leading_chunk(int S, int B, int Hkv, int ns, int cus) {
  int64_t chunks = WS_CUS / ((int64_t)B * Hkv * ((ns + 255) / 256));
  if (chunks > S / 128) chunks = S / 128;
  chunks = chunk_count(S, chunk_length(S, chunks)) / 2;
  const int64_t one_round = cus / ((int64_t)B * Hkv * ((ns + KEY_ROWS - 1) / KEY_ROWS));
  return chunk_length(S, chunks < one_round ? chunks : one_round);
}
// Floats of partial sums on any device: a smaller bound on the chunks never gives more of them, and a
// single chunk writes its results at once.
inline int64_t leading_floats(int S, int B, int Hkv, int ns) {
  const int chunks = chunk_count(S, leading_chunk(S, B, Hkv, ns, INT32_MAX));
  return chunks > 1 ? (int64_t)chunks * B * Hkv * ns * 2 * 128 : 0;
}

// The first ge.ns keys (LLM sinks; the text keys of the image patterns) against the queries of the
// whole sequence: every later query (CAUSAL) or every query.  set = chunk of ge.sink_chunk queries
// (leading_chunk on the host).  With several chunks the results are partial sums over the chunk.
// TWICE: for 64 leading keys at most, where a row block's second two wavefronts would have no rows.
// A step of such a workgroup then takes the time of one block instead of two: training steps with 64
// sinks, 32 / 8 heads, 504 -> 488 us (window 575, S = 8192), 830 -> 820 us (block Scatter G = 2, S = 6000).
template <bool CAUSAL, bool TWICE = false>
struct KeyRowsLeading {
  int S, ns, c0, c1;
  static IM_HD int num_sets(const IntraGeom& ge) { return (ge.S + ge.sink_chunk - 1) / ge.sink_chunk; }
  static IM_HD int max_rows(const IntraGeom& ge) { return TWICE ? 128 : im_min(ge.ns, ge.S); }
  IM_HD KeyRowsLeading(const IntraGeom& ge, int set, int) {
    S = ge.S;
    ns = im_min(ge.ns, ge.S);
    c0 = set * ge.sink_chunk;
    c1 = im_min(c0 + ge.sink_chunk, S);
  }
  IM_HD int n_rows() const { return TWICE ? 128 : ns; }
  IM_HD int n_cols() const { return S; }
  IM_HD int kpre() const { return 0; }
  IM_HD int row_pos(int t) const { return TWICE ? im_min(t & 63, ns - 1) : t; }  // (rows past the last key repeat it)
  IM_HD bool real(int t) const { return !TWICE || (t & 63) < ns; }
  IM_HD int col_pos(int c) const { return c; }
  IM_HD bool tile_at(int c, TileAt& a) const {
    a = TileAt{c, TILE_LINEAR};
    return true;
  }
  IM_HD int tile_rel(int, int i) const { return i; }
  IM_HD int lo(int t) const { return CAUSAL ? im_max(row_pos(t), c0) : c0; }
  IM_HD int hi(int) const { return c1 - 1; }
  IM_HD int block_lo(int r0, int) const { return lo(r0); }
  IM_HD int block_hi(int, int) const { return c1 - 1; }
  IM_HD bool store(int) const { return true; }
  static constexpr bool kEveryTile = true;
  static constexpr bool kBlockPredicate = false, kAccumulate = false;
  IM_HD bool sees(int, int) const { return true; }
};
using KeyRowsSinks = KeyRowsLeading<true>;
using KeyRowsFewSinks = KeyRowsLeading<true, true>;
using KeyRowsText = KeyRowsLeading<false>;
template <bool CAUSAL>
constexpr bool alternates<KeyRowsLeading<CAUSAL, true>> = true;

// Grid keys of group g of the image patterns (grid token (r, c) in group (r%2)*4 + c%4), against
// the queries of Scatter set g: its text chunk, then (unless TEXT_COLS_ONLY) its grid tokens; every
// pair is visible.  Scatter: dK / dV of the grid keys.  Gather 0: with TEXT_COLS_ONLY, what the text
// queries - which keep their Scatter rows - add to the grid keys' results of the window pass.
template <bool TEXT_COLS_ONLY>
struct KeyRowsImgGroup {
  MapImgScatter sc;
  static IM_HD int num_sets(const IntraGeom&) { return 8; }
  static IM_HD int max_rows(const IntraGeom& ge) { return ge.width * ge.width / 8; }
  static int longest(const IntraGeom& ge) { return KeyRowsImgGroup(ge, 0, 0).n_cols(); }  // (all row blocks of all groups)
  IM_HD KeyRowsImgGroup(const IntraGeom& ge, int set, int) : sc(ge, set, 0) {}
  IM_HD int n_rows() const { return sc.nimg; }
  IM_HD int n_cols() const { return TEXT_COLS_ONLY ? sc.chunk : sc.chunk + sc.nimg; }
  IM_HD int kpre() const { return 0; }
  IM_HD int row_pos(int t) const { return sc.imgpos(t); }
  IM_HD int col_pos(int c) const { return sc.qpos(c); }
  IM_HD bool tile_at(int c, TileAt& a) const { return sc.tile_in(c, sc.chunk, sc.chunk * sc.j, a); }
  IM_HD int tile_rel(int kind, int i) const { return sc.tile_rel(kind, i); }
  IM_HD int lo(int) const { return 0; }
  IM_HD int hi(int) const { return n_cols() - 1; }
  IM_HD int block_lo(int, int) const { return 0; }
  IM_HD int block_hi(int, int) const { return n_cols() - 1; }
  IM_HD bool store(int) const { return true; }
  static constexpr bool kEveryTile = false;
  static constexpr bool kBlockPredicate = false, kAccumulate = TEXT_COLS_ONLY;
  IM_HD bool sees(int, int) const { return true; }
};

// Grid keys of image Gather 0 against the grid queries.  Query patch (R, C) sees the grid rows
// win(R) .. win(R)+15 and columns win(C) .. win(C)+15, so key (r, c) is seen by whole 8x8 query
// patches: those with win(R) <= r < win(R)+16 and win(C) <= c < win(C)+16 - 2 x 2 of them away from
// the borders, and the same ones for all keys of an 8 x 8 square that starts half a patch (4 rows and
// 4 columns) from the patch grid.
// A set is one row block of up to 128 keys, its columns are the query patches that see any of them,
// 64 queries each, so a block of 32 columns lies inside one patch and a row meets all of it or
// nothing.  32 rows of the set (a wavefront) are a cell of 8 x 4 keys, half such a square, or of 4 x 8.
// Sets, in this order:
//  * for every s = 1 .. W/8 - 1 the 8 grid rows from 8s - 4 on: the 12 leftmost columns (a border cell
//    and a square), then 16 columns at a time (two squares: 2 x 3 patches of columns, of which a
//    wavefront works on its 4), up to the last 4 columns;
//  * the last 4 columns of these rows, 4 cells below each other at a time;
//  * the 4 upper and the 4 lower grid rows, 32 columns of the grid at a time: one patch row of columns.
// (Where W is an odd number of patches the runs of 16 columns end with one of 12 that holds the last 4.)
// (Behind the border, whose 12 rows or columns share a patch, a run streams more: rows or columns 12 ..
// 19 are seen by 3 patches, columns 12 .. 27 by 4, so that the longest row block has 3 x 4 of them - 3 x 5
// on a grid of 40 x 40, 4 x 4 on 32 x 32, where the other border is as near - and the mean one 6.2 to 7.)
// Runs of 16 columns from 0 on would stream 2 x 4 patches instead of 2 x 3, cells cut along the patches
// of the rows as well 3 x 4.
// No division by a variable past the constructor: col_pos and sees run several times per step.
struct KeyRowsImgWindow {
  int W, T, np, r0, c0, kw, wshift, wrows, wcols, Rlo, Clo, nR, nC, inv_nC;
  static IM_HD int mid_runs(const IntraGeom& ge) { return (ge.width + 8) / 16; }
  static IM_HD int side_runs(const IntraGeom& ge) { return ge.width % 16 == 0 ? (ge.width / 8 + 2) / 4 : 0; }
  static IM_HD int edge_runs(const IntraGeom& ge) { return (ge.width + 31) / 32; }
  static IM_HD int num_sets(const IntraGeom& ge) {
    return (ge.width / 8 - 1) * mid_runs(ge) + side_runs(ge) + 2 * edge_runs(ge);
  }
  static IM_HD int max_rows(const IntraGeom&) { return 128; }
  // (that of the rows and columns from 12 on, see above; two patches a side have one kind only)
  static int longest(const IntraGeom& ge) { return KeyRowsImgWindow(ge, ge.width > 16 ? mid_runs(ge) + 1 : 0, 0).n_cols(); }
  // first and last patch (along either axis) whose window covers grid row / column x
  static IM_HD int first_patch(int x) { return x <= 15 ? 0 : (x - 4) >> 3; }
  static IM_HD int last_patch(int x, int W) { return x >= W - 16 ? W / 8 - 1 : (x + 4) >> 3; }
  IM_HD KeyRowsImgWindow(const IntraGeom& ge, int set, int) {
    W = ge.width;
    T = ge.text_len;
    np = W / 8;
    const int mid = mid_runs(ge), n_mid = (np - 1) * mid, side = side_runs(ge);
    int height, cols;
    if (set < n_mid) {
      const int s = set / mid, run = set - s * mid;
      r0 = 8 * s + 4;
      c0 = run == 0 ? 0 : 16 * run - 4;
      height = 8;
      cols = run == 0 ? 12 : im_min(16, W - c0);
      kw = cols >> 2;
      wshift = 2;
      wrows = 0;
      wcols = 4;
    } else if (set < n_mid + side) {
      const int s = 4 * (set - n_mid);
      r0 = 8 * s + 4;
      c0 = W - 4;
      kw = im_min(4, np - 1 - s);
      height = 8 * kw;
      cols = 4;
      wshift = 2;
      wrows = 8;
      wcols = 0;
    } else {
      const int edge = edge_runs(ge), i = set - n_mid - side, e = i >= edge ? 1 : 0;
      r0 = e * (W - 4);
      c0 = (i - e * edge) * 32;
      height = 4;
      cols = im_min(32, W - c0);
      kw = cols >> 3;
      wshift = 3;
      wrows = 0;
      wcols = 8;
    }
    Rlo = first_patch(r0);
    Clo = first_patch(c0);
    nR = last_patch(r0 + height - 1, W) - Rlo + 1;
    nC = last_patch(c0 + cols - 1, W) - Clo + 1;
    inv_nC = 65535 / nC + 1;
  }
  IM_HD int n_rows() const { return 32 * kw; }
  IM_HD int n_cols() const { return 64 * nR * nC; }
  IM_HD int kpre() const { return 0; }
  IM_HD int patch_row(int pi) const { return (pi * inv_nC) >> 16; }  // pi / nC (exact: pi * nC < 2^16)
  IM_HD int key_r(int t) const { return r0 + (t >> 5) * wrows + ((t & 31) >> wshift); }
  IM_HD int key_c(int t) const { return c0 + (t >> 5) * wcols + (t & ((1 << wshift) - 1)); }
  IM_HD int row_pos(int t) const { return T + key_r(t) * W + key_c(t); }
  IM_HD int col_pos(int c) const {
    const int pi = c >> 6, u = c & 63;
    const int ri = patch_row(pi);
    return T + (8 * (Rlo + ri) + (u >> 3)) * W + 8 * (Clo + pi - ri * nC) + (u & 7);
  }
  IM_HD bool tile_at(int c, TileAt& a) const {
    a = TileAt{col_pos(c), TILE_PATCH};
    return true;
  }
  IM_HD int tile_rel(int, int i) const { return (i >> 3) * W + (i & 7); }
  IM_HD int lo(int) const { return 0; }
  IM_HD int hi(int) const { return n_cols() - 1; }
  IM_HD int block_lo(int, int) const { return 0; }
  IM_HD int block_hi(int, int) const { return n_cols() - 1; }
  IM_HD bool store(int) const { return true; }
  static constexpr bool kEveryTile = false;
  static constexpr bool kBlockPredicate = true, kAccumulate = false;
  IM_HD bool sees(int t, int c) const {
    const int pi = c >> 6, ri = patch_row(pi);
    const int wr = MapImgPatch::win_start(Rlo + ri, np), wc = MapImgPatch::win_start(Clo + pi - ri * nC, np);
    const int r = key_r(t), cc = key_c(t);
    return r >= wr && r < wr + 16 && cc >= wc && cc < wc + 16;
  }
};

}  // namespace intra
