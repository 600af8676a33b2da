// Backward kernels of the sparse attention for gfx950 (MI355X): dQ, dK and dV for the causal LLM
// patterns (Scatter, Gather 1, 64-aligned window, block Scatter with stripe offsets and sinks,
// per-token window with sinks) and the image patterns (Scatter, Gather 0).  Which rows meet which
// columns comes from the row maps of intra_bwd_maps.h.
//
// The reference has no backward kernels (its README names them as missing; training there runs
// through masked SDPA / FlexAttention, experiments/llm/llama_intra.py:26).  The math is the usual
//   P = exp(scale * S - lse),  dV = P^T dO,  dP = dO V^T,  dS = P o (dP - D),  D_i = dO_i . O_i,
//   dQ = scale * dS K,  dK = scale * dS^T Q.
//
// One template serves the three results, dQ in one launch and dK with dV in another.  A workgroup
// owns 256 / HP queries or 128 keys ("rows"; 32 per wavefront, held as MFMA B operands in registers
// like Q in the forward kernel) and streams the "columns" that see them through LDS in tiles of 64
// (K and V rows for dQ, Q and dO rows of every query head of the group for dK / dV).  Per 32
// columns a wavefront forms the scores S^T = C1 R1^T and dP^T = C2 R2^T, turns them into the
// weights (P or dS), packed to bf16 straight from the accumulators, and adds X^T W^T to its
// accumulators, X being the K, Q or dO tile read with transposing LDS reads - the data flow of
// the forward kernel without the online softmax.
#pragma once
#include <type_traits>

#include "intra_bwd_maps.h"
#include "intra_kernel.hip.h"

namespace intra {

// BWD_DKV forms dK and dV in one pass (the scores of a block are computed once for both): the two
// accumulators, the K and V fragments of the key rows, the scores, dP, both sets of weights and the
// operand ring need more than the 256 registers of a wavefront at two wavefronts per SIMD, so this
// mode runs workgroups of 4 wavefronts, one per SIMD, with up to 512 registers each.
// f(ic<B>{}), f(ic<B + 1>{}), ..., f(ic<E - 1>{})
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(ic<B>{});
    static_for<B + 1, E>(f);
  }
}

// BWD_DQ_HALF: dQ in half-size workgroups, 4 wavefronts of 128 / HP queries, two workgroups per CU, in steps of
// 32 columns (a ring of four half tiles).
enum BwdMode : int { BWD_DQ = 0, BWD_DKV = 1, BWD_DQ_HALF = 2 };
constexpr int bwd_waves(int mode) { return mode == BWD_DQ ? 8 : 4; }
static_assert(bwd_waves(BWD_DKV) * 32 == KEY_ROWS, "keys of a row block");

// Workgroups of one row map in a launch
struct BwdGrid {
  int n_rblocks;       // row blocks per set, or per part of one
  int hgroups;         // ratio / HP (dQ only)
  int items_per_pair;  // n_rblocks * hgroups
  int bundle;          // pairs of one XCD that are worked on together
  int blocks;          // workgroups, a multiple of 8
  int split;           // log2 of the parts that a pair's row blocks are split into (row block m: part m % 2^split), taken as pairs
};

struct BParams {
  const uint16_t *q, *k, *v, *o, *dout;  // bf16 (B, S, heads, 128)
  const float* lse;                      // (B, H, S): ln sum exp(scale * q.k) from the forward pass
  float* dsum;                           // (B, H, S) workspace: -D = -rowsum(dO o O), written by dQ, read by dK / dV
  float* l2;                             // (B, H, S) workspace: lse * log2(e), written by dQ, read by dK / dV
  uint16_t *dq, *dk, *dv;
  float* part;  // partial sums of the leading keys, dk then dv: (chunk, batch, kv head, key, 128) fp32
  // element strides: batch, row (token), head
  int64_t q_bs, q_rs, q_hs, k_bs, k_rs, k_hs, v_bs, v_rs, v_hs, o_bs, o_rs, o_hs, do_bs, do_rs, do_hs;
  int64_t dq_bs, dq_rs, dq_hs, dk_bs, dk_rs, dk_hs, dv_bs, dv_rs, dv_hs;
  int64_t lse_bs, lse_hs, lse_ts, ds_bs, ds_hs;  // dsum is contiguous over tokens
  int B, H, Hkv, ratio;
  int far_rows;      // some row of q, k, v or dout, or a token's workspace, is 4 GiB or more behind the first of its head
  IntraGeom geom;
  float scale;       // softmax scale
  float scale_log2;  // scale * log2(e)
  BwdGrid grid;      // the launch's row map
  BwdGrid lead;      // the leading keys that share the launch (blocks == 0: none)
  int lead_first;    // their workgroups come before the others
};

// two tiles and 2 x 64 column scalars, or two half tiles
constexpr int bwd_slot(int mode) { return mode == BWD_DQ_HALF ? 2 * FBLOCK32 : 2 * FTILE + 512; }
constexpr int bwd_ring_slots(int mode) { return mode == BWD_DQ ? 3 : 4; }
static_assert(2 * bwd_ring_slots(BWD_DQ_HALF) * bwd_slot(BWD_DQ_HALF) <= 160 * 1024, "two workgroups per CU");

// 64 lanes x 4 bytes from per-lane global addresses to 256 consecutive LDS bytes at lds_addr (the
// active lanes' parts of them), like dma_group
__device__ __forceinline__ void dma_dwords(const void* gsrc, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(gsrc), "s"(lds_addr) : "memory");
}

// The same two with a wave-uniform address and 32-bit per-lane byte offsets
template <int LDS_OFFSET>
__device__ __forceinline__ void dma_rows(const void* base, uint32_t offset, uint32_t lds_addr) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               : : "v"(offset), "s"(base), "s"(lds_addr), "n"(LDS_OFFSET) : "memory", "scc");
}
template <int LDS_OFFSET>
__device__ __forceinline__ void dma_scalars(const void* base, uint32_t offset, uint32_t lds_addr) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
               : : "v"(offset), "s"(base), "s"(lds_addr), "n"(LDS_OFFSET) : "memory", "scc");
}

// The work of one workgroup, number `block` of the grid `g`.  RMAP: row map (intra_bwd_maps.h).
// PARTIAL: where there are several sets, the results are partial sums over the set's columns, written
// as fp32 to p.part instead of bf16 to dk / dv (leading keys).  FAR: the columns are requested by 64-bit
// addresses.
//
// MFMA layout (v_mfma_f32_16x16x32_bf16, as in the forward kernel): a block of 32 columns times the
// wavefront's 32 rows is 2 x 2 tiles [ct][rt] with 4 k-steps; lane (l16 = lane % 16, g4 = lane / 16)
// holds columns 16*ct + 4*g4 .. +3 of row 16*rt + l16.  The packed weights of a row tile are the B
// operand of the accumulation, whose 32-column reduction is numbered slot s of lane quarter g4 =
// column 16*(s/4) + 4*g4 + s%4; the transposing reads of the X tile follow that numbering.
template <class RMAP, int MODE, int HP, bool PARTIAL, bool FAR>
__device__ __forceinline__ void bwd_rows(const BParams& p, const BwdGrid& g, const int block, unsigned char* const smem) {
  constexpr int NW = bwd_waves(MODE);
  constexpr bool ROWS_ARE_QUERIES = MODE != BWD_DKV;
  constexpr bool HALF = MODE == BWD_DQ_HALF;  // a step is one block of 32 columns
  constexpr int BWD_SLOT = bwd_slot(MODE);
  constexpr int SECOND = HALF ? FBLOCK32 : FTILE;  // the second tile of a slot
  constexpr int POS = ROWS_ARE_QUERIES ? NW * 32 / HP : NW * 32;  // rows per row block (of one head)

  // BWD_DKV: a step of its single wavefront per SIMD is about as long as a tile takes to arrive, so
  // its ring is one slot deeper and a tile has two steps to land; the column scalars travel the same
  // way instead of through registers.  BWD_DQ_HALF has the same ring of half tiles.
  constexpr bool DEEP = MODE != BWD_DQ;
  // BWD_DKV's wavefront is alone on its SIMD: nothing covers what it issues between its blocks.  So the requests of a
  // step (three instructions each, nine of them) go behind MFMAs of its first block, and which blocks of a tile it
  // needs and whether any of their pairs are hidden is worked out once per tile, not per head.  Training steps, in
  // one piece in front of the blocks / so, us: Scatter G=8 S=32768 4339 / 4243, window 575 with 64 sinks S=8192 448 / 436,
  // block Scatter S=6000 with 64 sinks 712 / 687, image Gather 0 1024^2 309 / 309.  (Left out altogether, of a
  // Scatter step of 4265 us: without the requests 4233, the transposing reads 4231, all vector instructions 4168.  What
  // remains is the MFMAs, at the clock that the board's power allows.)
  constexpr bool SPREAD = MODE == BWD_DKV && !FAR;
  constexpr bool ALT = alternates<RMAP>;  // wavefronts 0, 1 and 2, 3 share rows and take turns at the 32-column blocks
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15;
  const int g4 = lane >> 4;

  // ---------------------------------------------------------------- work item
  // Workgroups start in blockIdx order, round-robin over the 8 XCDs, and a CU takes the next one
  // when it has finished one (half-size ones: when it has finished one of its two).  The unit is a part of a (set, batch,
  // kv head) pair: all its row blocks, or every 2nd, 4th or 8th where whole pairs would leave XCDs idle (xcd_split).
  // Per XCD the parts are taken in bundles of `bundle`, as few as fill its 32 CUs (64 places for half-size workgroups), so
  // that the workgroups running together stream the same few megabytes of columns through the XCD's L2, or all as one
  // bundle where the last one's long row blocks would end the launch late (one_bundle_pays).  Within a bundle the row
  // blocks with the most columns come first (the last query blocks for dQ, the first key blocks for dK / dV).
  const int xcd = block & 7, slot = block >> 3;
  const int per_bundle = g.bundle * g.items_per_pair;
  const int bun = slot / per_bundle, rem = slot - bun * per_bundle;
  const int heavy = rem / g.bundle;
  const int nbh = p.B * p.Hkv;
  const int part = (bun * g.bundle + (rem - heavy * g.bundle)) * 8 + xcd;
  const int pair = part >> g.split;
  if (pair >= RMAP::num_sets(p.geom) * nbh) return;
  int hg = 0, rblk = heavy;
  if (ROWS_ARE_QUERIES) {
    hg = heavy % g.hgroups;
    rblk = g.n_rblocks - 1 - heavy / g.hgroups;
  }
  rblk = (rblk << g.split) + (part - (pair << g.split));
  const int set = pair / nbh;
  const int bh = pair % nbh;
  const int batch = bh / p.Hkv;
  const int kvh = bh % p.Hkv;

  const int r0 = rblk * POS;
  const RMAP map(p.geom, set, r0);
  const int kpre = map.kpre();
  const int n_rows = map.n_rows(), n_cols = map.n_cols();
  if (r0 >= n_rows) return;
  const int r1 = im_min(r0 + POS, n_rows) - 1;

  // Row r meets the columns lo(r)..hi(r) (plus those below kpre for maps that have such a prefix).
  const int cb = map.block_lo(r0, r1);  // first column of the row block
  const int ce = map.block_hi(r0, r1);  // last one
  const int ntiles = ce >= cb ? (ce - cb + BN) / BN : 0;

  // ---------------------------------------------------------------- this wavefront's rows
  // a lane works for two rows: 16 * rt + l16 of the wavefront's 32 (rows past the end repeat the last)
  const int hw = ROWS_ARE_QUERIES ? wave % HP : 0;
  const int wr0 = r0 + (ROWS_ARE_QUERIES ? wave / HP : wave) * 32;
  const bool wave_active = wr0 <= r1;
  bool row_valid[2];
  int row[2], lo_l[2], hi_l[2];
  int64_t rpos[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    row_valid[rt] = wr0 + 16 * rt + l16 <= r1;
    row[rt] = im_min(wr0 + 16 * rt + l16, r1);
    lo_l[rt] = map.lo(row[rt]);
    hi_l[rt] = map.hi(row[rt]);
    if constexpr (ALT) row_valid[rt] = row_valid[rt] && map.real(row[rt]);
    rpos[rt] = map.row_pos(row[rt]);
  }
  // union and intersection of the ranges of the wavefront's rows
  WaveBounds wb;
  {
    int a = im_min(lo_l[0], lo_l[1]), b = im_max(hi_l[0], hi_l[1]), c = im_max(lo_l[0], lo_l[1]), d = im_min(hi_l[0], hi_l[1]);
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) {
      a = im_min(a, __shfl_xor(a, m));
      b = im_max(b, __shfl_xor(b, m));
      c = im_max(c, __shfl_xor(c, m));
      d = im_min(d, __shfl_xor(d, m));
    }
    wb.w_lo = __builtin_amdgcn_readfirstlane(a);
    wb.w_hi = __builtin_amdgcn_readfirstlane(b);
    wb.f_lo = __builtin_amdgcn_readfirstlane(c);
    wb.f_hi = __builtin_amdgcn_readfirstlane(d);
  }
  // The blocks of 32 columns (counted from cb) that this wavefront's rows meet: one range; with a
  // prefix it starts at the first block (the main loop skips those between prefix and own range).
  const bool any = wave_active && wb.w_hi >= cb && (kpre > 0 || wb.w_hi >= wb.w_lo);  // (early rows may meet prefix columns only)
  const int jb_lo = !any ? 1 : kpre > 0 ? 0 : (im_max(wb.w_lo, cb) - cb) >> 5;
  const int jb_hi = !any ? 0 : (wb.w_hi - cb) >> 5;
  const int hq = kvh * p.ratio + hg * HP + hw;  // query head of a query row

  // ---------------------------------------------------------------- row operands (MFMA B fragments)
  // [rt][ks]: lane holds row 16 * rt + l16, head dims 32 * ks + 8 * g4 .. +7
  bf16x8 r1f[2][4], r2f[2][4];
  float L2_row[2] = {0.f, 0.f}, D_row[2] = {0.f, 0.f};
  // kAccumulate: the result rows as an earlier pass wrote them, in the layout of store_rows.  Requested with
  // the operands: read one by one in front of the stores they were 16 round trips behind each other (image
  // Gather 0 training step, 24 heads: 1346 -> 1315 us at 2048^2).
  const int chunk_ofs = (2 * (g4 & 1) + (g4 >> 1)) * 8;  // the lane's 8 of every 32 head dims of a result row
  u32x4 old_k[RMAP::kAccumulate ? 2 : 1][4], old_v[RMAP::kAccumulate ? 2 : 1][4];
  auto load_rows = [&] {
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const uint16_t *a1, *a2;
    if (ROWS_ARE_QUERIES) {
      a1 = p.q + (batch * p.q_bs + rpos[rt] * p.q_rs + hq * p.q_hs + g4 * 8);
      a2 = p.dout + (batch * p.do_bs + rpos[rt] * p.do_rs + hq * p.do_hs + g4 * 8);
    } else {
      a1 = p.k + (batch * p.k_bs + rpos[rt] * p.k_rs + kvh * p.k_hs + g4 * 8);
      a2 = p.v + (batch * p.v_bs + rpos[rt] * p.v_rs + kvh * p.v_hs + g4 * 8);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      r1f[rt][ks] = *reinterpret_cast<const bf16x8*>(a1 + ks * 32);
      r2f[rt][ks] = *reinterpret_cast<const bf16x8*>(a2 + ks * 32);
    }
    if constexpr (RMAP::kAccumulate) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        old_k[rt][m] = *reinterpret_cast<const u32x4*>(p.dk + (batch * p.dk_bs + rpos[rt] * p.dk_rs + kvh * p.dk_hs + chunk_ofs + 32 * m));
        old_v[rt][m] = *reinterpret_cast<const u32x4*>(p.dv + (batch * p.dv_bs + rpos[rt] * p.dv_rs + kvh * p.dv_hs + chunk_ofs + 32 * m));
      }
    }
    if (ROWS_ARE_QUERIES) {
      // D = dO . O of the row: this lane's 32 head dims, then the rest from the other three lanes of the row
      const uint16_t* ao = p.o + (batch * p.o_bs + rpos[rt] * p.o_rs + hq * p.o_hs + g4 * 8);
      float part = 0.f;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const bf16x8 of = *reinterpret_cast<const bf16x8*>(ao + ks * 32);
#pragma unroll
        for (int d = 0; d < 8; ++d) part += (float)r2f[rt][ks][d] * (float)of[d];
      }
      D_row[rt] = lane_quad_sum(part);
      L2_row[rt] = p.lse[batch * p.lse_bs + hq * p.lse_hs + rpos[rt] * p.lse_ts] * 1.4426950408889634f;
      if (row_valid[rt] && g4 == 0) {  // what the dK / dV launches need per query, in the form they use it
        p.dsum[batch * p.ds_bs + hq * p.ds_hs + rpos[rt]] = -D_row[rt];
        p.l2[batch * p.ds_bs + hq * p.ds_hs + rpos[rt]] = L2_row[rt];
      }
    }
  }
  };
  if (!DEEP) load_rows();  // (the deep ring requests its first tiles before them, see below)

  // ---------------------------------------------------------------- LDS addressing (as in the forward kernel)
  const int ld_row = lane >> 4;
  const uint32_t ld_col = (((lane & 15) ^ (4 * ld_row)) << 4);
  int kaddr[4];
  {
    const int r = l16 & 3;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) kaddr[ks] = (l16 >> 2) * FGROUP_STRIDE + r * 256 + 64 * (ks ^ r) + 16 * g4;
  }
  int vaddr[4];
  {
    const int ri = l16 >> 2;
#pragma unroll
    for (int a = 0; a < 4; ++a)
      vaddr[a] = g4 * FGROUP_STRIDE + ri * 256 + 64 * (a ^ ri) + 16 * ((l16 & 3) >> 1) + 8 * (l16 & 1);
  }
  // LDS operands are read from per-lane bases that carry the ring slot (b0: the step's slot, b1: the
  // next one's), advanced once per step, so that everything else is a compile-time offset.
  // kread_b: row-per-lane operand 2 * ks + ct of a 32-row block (rows 16 * ct + l16, head dims of
  // k-step ks); vread_b: transposed operand (head dims 16 * dt .. + 15 of the block's 32 rows).
  // sb0, sb1: the same for the column scalars of the deep ring.
  // (Wavefronts that take turns at the blocks work on one block of a tile; theirs is in the bases.)
  const int half = ALT ? wave >> 1 : 0;
  int kb0[4], kb1[4], vb0[4], sb0 = 0, sb1 = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    kb0[i] = half * FBLOCK32 + kaddr[i];
    kb1[i] = half * FBLOCK32 + BWD_SLOT + kaddr[i];
    vb0[i] = half * FBLOCK32 + vaddr[i];
  }
  sb0 = 2 * FTILE + 128 * half + 16 * g4;
  sb1 = BWD_SLOT + 2 * FTILE + 128 * half + 16 * g4;
  auto kread_b = [&](const int (&kb)[4], int off, int f) {
    return *reinterpret_cast<const bf16x8*>(smem + (kb[f >> 1] + (off + (f & 1) * 4 * FGROUP_STRIDE)));
  };
  auto vread_b = [&](int off, int dt) {
    const int o2 = vb0[dt >> 1] + (off + 32 * (dt & 1));
    bf16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(smem + o2));
    bf16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (__attribute__((address_space(3))) bf16x4*)(smem + (o2 + 4 * FGROUP_STRIDE)));
    return __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto mfma = [](bf16x8 a, bf16x8 b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); };
  const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};

  floatx4 acc[8][2];  // [head-dim tile][row tile]: head dims 16 * dt + 4 * g4 .. + 3 of row 16 * rt + l16
  floatx4 acc_v[MODE == BWD_DKV ? 8 : 1][2];  // BWD_DKV: dV (acc is dK)
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      acc[dt][rt] = zero4;
      if (MODE == BWD_DKV) acc_v[dt][rt] = zero4;
    }
  const float c2 = p.scale_log2;
  const float s_hidden = c2 >= 0.f ? -INFINITY : INFINITY;  // score that gives exp2(s * c2 - lse) = 0

  // ---------------------------------------------------------------- column steps
  // dQ meets one stream of columns (the K / V rows of the kv head), tile after tile from the first.
  // dK / dV meet one per query head of the group (its Q / dO rows); they take the tiles from the
  // last one down and, per tile, head after head: all key blocks of a (set, batch, kv head) start
  // at the last tile together and stay in step, so that a tile fetched for one of them is in the
  // L2 for the others.  A step is one (tile, head).
  const int n_streams = ROWS_ARE_QUERIES ? 1 : p.ratio;
  const int n_steps = HALF ? (ce >= cb ? (ce - cb + 32) >> 5 : 0) : ntiles * n_streams;
  struct Cursor {
    int tile, head;
  };
  auto advance = [&](Cursor& c) {
    if (ROWS_ARE_QUERIES) {  // (HALF: half tiles)
      ++c.tile;
    } else if (++c.head == n_streams) {
      c.head = 0;
      --c.tile;
    }
  };
  const char *c1base, *c2base;
  uint32_t c1rs, c2rs;
  int64_t c1hs = 0, c2hs = 0;  // byte stride between the heads of the group (dK / dV)
  if (ROWS_ARE_QUERIES) {
    c1base = reinterpret_cast<const char*>(p.k + batch * p.k_bs + kvh * p.k_hs);
    c2base = reinterpret_cast<const char*>(p.v + batch * p.v_bs + kvh * p.v_hs);
    c1rs = (uint32_t)(p.k_rs * 2);
    c2rs = (uint32_t)(p.v_rs * 2);
  } else {
    c1base = reinterpret_cast<const char*>(p.q + batch * p.q_bs + kvh * p.ratio * p.q_hs);
    c2base = reinterpret_cast<const char*>(p.dout + batch * p.do_bs + kvh * p.ratio * p.do_hs);
    c1rs = (uint32_t)(p.q_rs * 2);
    c2rs = (uint32_t)(p.do_rs * 2);
    c1hs = p.q_hs * 2;
    c2hs = p.do_hs * 2;
  }
  // Requests.  A lane's rows of a tile are named by 32-bit byte offsets from a wave-uniform address.  For
  // tiles whose positions follow one of the maps' patterns (tile_at) the offsets stay in registers from
  // tile to tile and only that address moves; a tile cut by the end of the columns (its last row repeated)
  // and, in maps whose tiles do not all follow a pattern, the others get offsets of their own.  The query
  // heads of a group share the offsets.  With the addresses worked out per lane and request (a 64-bit
  // multiply-add each, behind a 64-bit product for the head's base) a step of dK / dV issued about 120
  // instructions for its requests, none of them behind an MFMA.  With these and the order of the block below
  // (same box, training steps, us): Scatter G=8 S=32768 4385 -> 4189, its dK / dV launch 2395 -> 2090; image
  // Scatter 2048^2 at 12 heads 1166 -> 1076; window 575 with 64 sinks, S=8192, 486 -> 470; image Gather 0
  // 1024^2 363 -> 344.
  // What ordinary calls do not need stays out of the step, whose scalar registers are few: tensors beyond
  // the reach of 32-bit offsets have kernels of their own (FAR; inlined here, their addresses kept 10 - 24
  // scalars in lanes of vector registers), maps whose every tile follows a pattern (kEveryTile) hold no
  // code for positions key by key, and the ring's slots follow from the present one.  Scalars moved to
  // lanes and back on the ordinary path of a step: block Scatter 16 -> 1, Scatter 4 -> 0.  Training steps, us:
  // block Scatter S=6000 780.5 -> 764.9, window 575 with 64 sinks, S=8192, 476.2 -> 468.9.
  constexpr int GROUPS = 16 / NW;  // 4-row groups of either tile per wavefront
  constexpr int STEP_GROUPS = HALF ? GROUPS / 2 : GROUPS;  // those of a step (HALF: one half of the tile, then the other)
  // first row of group gi of this wavefront in the tile
  auto group_row = [&](int gi) { return 4 * (wave * STEP_GROUPS + gi % STEP_GROUPS) + 32 * (gi / STEP_GROUPS) + ld_row; };
  uint32_t vo1[GROUPS], vo2[GROUPS], vos = 0;
#pragma unroll
  for (int gi = 0; gi < GROUPS; ++gi) vo1[gi] = vo2[gi] = 0;
  int vo_kind = -1;                     // what the offsets are for: a tile pattern, or -1
  const char *a1 = c1base, *a2 = c2base, *as = nullptr;  // addresses of the step being requested
  // the column scalars that this wavefront requests: lse * log2(e) (even wavefronts) or -D
  const float* const sbase = (wave & 1 ? p.dsum : p.l2) + (batch * p.ds_bs + kvh * p.ratio * p.ds_hs);
  auto aim = [&](int tile) {  // at the first head of a tile
    const int c = cb + tile * BN;
    const int last = n_cols - 1 - c;
    const bool cut = last < BN - 1;
    TileAt at;
    const bool pattern = (RMAP::kEveryTile || !cut) && map.tile_at(c, at);
    if (RMAP::kEveryTile || pattern) {
      if (vo_kind != at.kind || (RMAP::kEveryTile && cut)) {
        vo_kind = RMAP::kEveryTile && cut ? -1 : at.kind;
        auto row_of = [&](int i) { return (uint32_t)map.tile_rel(at.kind, RMAP::kEveryTile ? im_min(i, last) : i); };
#pragma unroll
        for (int gi = 0; gi < GROUPS; ++gi) {
          const uint32_t rel = row_of(group_row(gi));
          vo1[gi] = rel * c1rs + ld_col;
          vo2[gi] = rel * c2rs + ld_col;
        }
        if (!ROWS_ARE_QUERIES) vos = 4 * row_of(lane);
      }
    } else {
      vo_kind = -1;
      at.base = 0;
#pragma unroll
      for (int gi = 0; gi < GROUPS; ++gi) {
        const uint32_t pos = (uint32_t)map.col_pos(im_min(c + group_row(gi), n_cols - 1));
        vo1[gi] = pos * c1rs + ld_col;
        vo2[gi] = pos * c2rs + ld_col;
      }
      if (!ROWS_ARE_QUERIES) vos = 4 * (uint32_t)map.col_pos(im_min(c + lane, n_cols - 1));
    }
    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane(at.base);
    a1 = c1base + (uint64_t)base * c1rs;
    a2 = c2base + (uint64_t)base * c2rs;
    if (!ROWS_ARE_QUERIES) as = reinterpret_cast<const char*>(sbase + base);
  };
  const uint32_t lds_rows = lds_base + wave * STEP_GROUPS * FGROUP_STRIDE;
  const uint32_t lds_scalars = lds_base + 256 * (wave & 1);
  constexpr int REQUESTS = 2 * STEP_GROUPS + (ROWS_ARE_QUERIES ? 0 : 1);  // per wavefront and step
  // request n of a step of dK / dV: the groups of either tile in turns, then the scalars (wavefronts 2, 3 repeat
  // those of 0, 1: every wavefront counts alike)
  auto request_one = [&](auto n_c, int slot_off) {
    constexpr int n = decltype(n_c)::value;
    if constexpr (n == 2 * GROUPS) dma_scalars<2 * FTILE>(as, vos, lds_scalars + slot_off);
    else if constexpr (n % 2 == 0) dma_rows<n / 2 * FGROUP_STRIDE>(a1, vo1[n / 2], lds_rows + slot_off);
    else dma_rows<FTILE + n / 2 * FGROUP_STRIDE>(a2, vo2[n / 2], lds_rows + slot_off);
  };
  auto load_step = [&](const Cursor& cu, int slot_off) {
    const int tile = HALF ? cu.tile >> 1 : cu.tile;
    if constexpr (FAR) {
      const int c = cb + cu.tile * (HALF ? 32 : BN);
#pragma unroll
      for (int gi = 0; gi < STEP_GROUPS; ++gi) {
        const uint64_t pos = (uint64_t)map.col_pos(im_min(c + group_row(gi), n_cols - 1));
        dma_group(c1base + (cu.head * c1hs + pos * c1rs + ld_col), lds_rows + slot_off + gi * FGROUP_STRIDE);
        dma_group(c2base + (cu.head * c2hs + pos * c2rs + ld_col), lds_rows + slot_off + SECOND + gi * FGROUP_STRIDE);
      }
      if (!ROWS_ARE_QUERIES)
        dma_dwords(sbase + (cu.head * p.ds_hs + map.col_pos(im_min(c + lane, n_cols - 1))),
                   lds_scalars + slot_off + 2 * FTILE);
      return;
    }
    if constexpr (SPREAD) {
      if (cu.head == 0) {
        aim(tile);
      } else {  // from one head's addresses to the next one's
        a1 += c1hs;
        a2 += c2hs;
        as += 4 * (uint32_t)p.ds_hs;  // (S floats)
      }
      if (slot_off >= 0) static_for<0, REQUESTS>([&](auto n_c) { request_one(n_c, slot_off); });
      return;
    }
    if (HALF ? (cu.tile & 1) == 0 : true) aim(tile);
    auto request = [&](auto first_c) {  // the groups from `first` on
      static_for<0, STEP_GROUPS>([&](auto gi_c) {
        constexpr int gi = decltype(gi_c)::value, first = decltype(first_c)::value;
        dma_rows<gi * FGROUP_STRIDE>(a1, vo1[first + gi], lds_rows + slot_off);
        dma_rows<SECOND + gi * FGROUP_STRIDE>(a2, vo2[first + gi], lds_rows + slot_off);
      });
    };
    if (HALF && (cu.tile & 1)) request(ic<HALF ? STEP_GROUPS : 0>{});
    else request(ic<0>{});
  };
  // Three tile slots: while step t works on its tile, the tile of step t+1 has landed (the scores
  // of its first block are formed at the end of step t) and the tile of step t+2 is in flight.
  Cursor cur{ROWS_ARE_QUERIES ? 0 : ntiles - 1, 0};  // step being computed
  Cursor ld = cur;                                   // step being requested
  // (Deep ring: one slot more, the tile of step t+3 is requested during step t, and the barrier of a step leaves the
  // requests of the step before in flight.  SPREAD: every step makes as many, the last three for a tile that nobody
  // reads, and the wait behind the loop is for these.  Otherwise the last steps make none, and the barriers behind them
  // wait for all.)
  for (int t = 0; t < (DEEP ? 3 : 2) && t < n_steps; ++t) {
    if (SPREAD && t > 0) advance(ld);  // (SPREAD: ld is the step requested last)
    load_step(ld, t * BWD_SLOT);
    if (!SPREAD) advance(ld);
  }
  // The deep ring's barriers leave requests in flight.  The row operands are ordinary loads the
  // compiler waits for at their first use, inside the main loop, with a count that knows nothing of
  // the requests issued by hand - it would wait for those as well, every time round.  So they are
  // requested here, behind the first tiles (whose latency they share), and land here, once.
  if (DEEP) {
    load_rows();
    __builtin_amdgcn_s_waitcnt((0 & 15) | (7 << 4) | (15 << 8) | (0 << 14));  // vmcnt(0)
    // They stay in the accumulation half of the register file, where an MFMA reads its B operand as well.  Of
    // its own accord the compiler puts nothing but accumulators there, and copied them, or the V fragments,
    // between the halves inside the blocks: of few sinks 44 moves and 13 waiting instructions per 64 MFMAs.
    // With this no block holds a move (training step, window 575 with 64 sinks, S=8192, us: 471.3 -> 467.2).
    if constexpr (!ROWS_ARE_QUERIES)
#pragma unroll
    for (int i = 0; i < 8; ++i) asm volatile("" : "+a"(r1f[i >> 2][i & 3]), "+a"(r2f[i >> 2][i & 3]));
  }
  constexpr int LAST_SLOT = (bwd_ring_slots(MODE) - 1) * BWD_SLOT;
  int ring = 0;  // slot of the step being computed
  auto slot_after = [](int s) { return s == LAST_SLOT ? 0 : s + BWD_SLOT; };
  bool fresh = n_steps >= 3;  // the most recent request is for the step after the next
  floatx4 s_cur[2][2];  // [ct][rt]
#pragma unroll
  for (int t = 0; t < 4; ++t) s_cur[t >> 1][t & 1] = zero4;
  bool have = false;  // s_cur and fr hold what a previous block prepared for the one that comes next
  // One slot is one MFMA; an LDS operand serves two consecutive slots (the two row tiles).
  constexpr int NFRAG = MODE == BWD_DKV ? 32 : 24;  // LDS operands per block
  constexpr int LA = MODE == BWD_DKV ? 8 : 4;       // operands between the request of one and its use
  static_assert(NFRAG % LA == 0, "a block must leave the ring where the next block expects it");
  bf16x8 fr[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) fr[i] = bf16x8{};
  floatx4 l4_keep[2] = {zero4, zero4}, d4_keep[2] = {zero4, zero4};
  // dQ: -D of the lane's two rows, as the accumulators of dP start from it
  const floatx4 nd_row[2] = {floatx4{-D_row[0], -D_row[0], -D_row[0], -D_row[0]}, floatx4{-D_row[1], -D_row[1], -D_row[1], -D_row[1]}};
  // (dK / dV without a block predicate: what the wavefront does with the blocks of a tile, worked out once for all heads)
  constexpr bool PER_TILE = SPREAD && !RMAP::kBlockPredicate;
  int todo = 0;  // bits 2 * blk: the block is wanted, 2 * blk + 1: none of it is hidden
  for (int t = 0; t < n_steps; ++t) {
    // the tiles of steps t and t+1 have landed for everybody; nobody reads that of t-1
    if (SPREAD || (DEEP && fresh)) tile_barrier<REQUESTS>();
    else tile_barrier<0>();
    // the tile of step t + 3 (BWD_DQ: t + 2) into the slot of step t - 1
    const int free_slot = ring == 0 ? LAST_SLOT : ring - BWD_SLOT;
    if constexpr (SPREAD) {
      // Behind the last steps the last tile is requested again, which nobody reads: every step leaves the same number
      // of requests in flight.
      if (t + 3 < n_steps) {
        advance(ld);
        load_step(ld, -1);
      }
    } else {
      fresh = t + (DEEP ? 3 : 2) < n_steps;
      if (fresh) {
        load_step(ld, free_slot);
        advance(ld);
      }
    }
    if (PER_TILE && cur.head == 0) {
      todo = 0;
#pragma unroll
      for (int blk = 0; blk < (ALT ? 1 : 2); ++blk) {
        const int jb = 2 * cur.tile + (ALT ? half : blk);
        const int sb_lo = cb + 32 * jb;
        if (jb >= jb_lo && jb <= jb_hi && (kpre == 0 || block_wanted(wb, kpre, sb_lo))) todo |= 1 << (2 * blk);
        if (block_unmasked(wb, kpre, sb_lo)) todo |= 2 << (2 * blk);
      }
    }
    static_for<0, ALT || HALF ? 1 : 2>([&](auto blk_c) {
      constexpr int blk = decltype(blk_c)::value;
      const int jb = HALF ? cur.tile : 2 * cur.tile + (ALT ? half : blk);
      const int sb_lo = cb + 32 * jb;  // first column of the block
      // (behind the prefix and in front of the wavefront's own range nothing is visible: a run of 4 image
      // patches streams 10 tiles of window keys, of which a patch sees 4: training steps of 24 heads
      // 397 -> 392 us at 1024^2, 1259 -> 1236 us at 2048^2)
      bool wanted = PER_TILE ? (todo >> (2 * blk)) & 1 : jb >= jb_lo && jb <= jb_hi && (kpre == 0 || block_wanted(wb, kpre, sb_lo));
      // maps with a block predicate: a row meets the whole block or nothing of it
      bool lane_sees[2] = {true, true};
      bool masked;
      if constexpr (RMAP::kBlockPredicate) {
        lane_sees[0] = map.sees(row[0], sb_lo);
        lane_sees[1] = map.sees(row[1], sb_lo);
        wanted = wanted && __builtin_amdgcn_ballot_w64(lane_sees[0] || lane_sees[1]) != 0;
        masked = __builtin_amdgcn_ballot_w64(lane_sees[0] && lane_sees[1]) != ~0ull;
      } else {
        masked = PER_TILE ? !((todo >> (2 * blk + 1)) & 1) : !block_unmasked(wb, kpre, sb_lo);
      }
      constexpr bool REQUEST = SPREAD && blk == 0;
      if constexpr (REQUEST) {
        // (A branch of its own: with this code in the way around the block the compiler gives the accumulators other
        // registers and moves them in and out of the block.)
        int w = __builtin_amdgcn_readfirstlane((int)wanted);
        asm volatile("" : "+s"(w));
        if (!w) static_for<0, REQUESTS>([&](auto n_c) { request_one(n_c, free_slot); });
        asm volatile("" : "+s"(w));
        wanted = w;
      }
      if (!wanted) {
        have = false;
        return;
      }
      // Hand-scheduled.  Slots 0-15: dP of this block, 16-31: the scores of the next block, then the
      // accumulation (dQ), or those of dV (32-47) and dK (48-63).  LDS operand f (slots 2f, 2f+1) is
      // requested LA operands earlier into a ring of LA fragments, across block and step boundaries (both
      // following blocks have landed).  What a slot may hold besides its MFMA was found with isolated
      // loops on one SIMD: an MFMA keeps the vector port for 8 of its 16 cycles, so 8 cycles of vector
      // work behind it (two plain instructions or one exponential) cost nothing and the rest does, and a
      // request or a wait costs nothing directly behind the MFMA but some 10 cycles in front of one.
      // Hence one exponential or two plain instructions per slot, and MFMA, wait, request, vector work in
      // that order; sched_barrier keeps the compiler from regrouping.
      auto fetch = [&](int f) {
        const int here = blk * FBLOCK32;  // the block inside the step's slot
        // rows of the block that follows in this order, at tile `which` of its slot
        auto next_rows = [&](int which, int ff) {
          if (ALT || HALF) return kread_b(kb1, which * SECOND, ff);
          return blk == 0 ? kread_b(kb0, FBLOCK32 + which * SECOND, ff) : kread_b(kb1, which * SECOND, ff);
        };
        if (MODE == BWD_DKV) {
          if (f < 8) return kread_b(kb0, here + FTILE, f);   // dO rows: dP
          if (f < 16) return next_rows(0, f - 8);            // Q rows of the next block: its scores
          if (f < 24) return vread_b(here + FTILE, f - 16);  // dO^T: dV accumulation
          if (f < 32) return vread_b(here, f - 24);          // Q^T: dK accumulation
          return next_rows(1, f - 32);
        }
        if (f < 8) return kread_b(kb0, here + SECOND, f);
        if (f < 16) return next_rows(0, f - 8);
        if (f < 24) return vread_b(here, f - 16);
        return next_rows(1, f - 24);
      };
      const float* sc = reinterpret_cast<const float*>(smem + (sb0 + 128 * blk));
      // scalars of the block that follows in this order
      const float* scn = ALT ? reinterpret_cast<const float*>(smem + sb1) : blk == 0 ? sc + 32 : reinterpret_cast<const float*>(smem + sb1);
      if (!have) {  // first block of a run: nothing was prepared by a previous block
        if (MODE == BWD_DKV) {
          l4_keep[0] = *reinterpret_cast<const floatx4*>(sc);
          l4_keep[1] = *reinterpret_cast<const floatx4*>(sc + 16);
          d4_keep[0] = *reinterpret_cast<const floatx4*>(sc + 64);
          d4_keep[1] = *reinterpret_cast<const floatx4*>(sc + 64 + 16);
        }
#pragma unroll
        for (int t4 = 0; t4 < 4; ++t4) s_cur[t4 >> 1][t4 & 1] = zero4;
#pragma unroll
        for (int f = 0; f < 8; ++f) {
          const bf16x8 a = kread_b(kb0, blk * FBLOCK32, f);
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) s_cur[f & 1][rt] = mfma(a, r1f[rt][f >> 1], s_cur[f & 1][rt]);
        }
#pragma unroll
        for (int i = 0; i < LA; ++i) fr[i] = fetch(i);
      }
      if (masked) {  // scores of invisible pairs become -inf (for a positive scale): weight 0
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
          for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const bool vis = RMAP::kBlockPredicate ? lane_sees[rt]
                                                     : key_visible(sb_lo + 16 * ct + 4 * g4 + e, kpre, lo_l[rt], hi_l[rt]);
              if (!vis) s_cur[ct][rt][e] = s_hidden;
            }
      }
      floatx4 dp[2][2], s_next[2][2];
      bf16x8 wp[2];
      bf16x8 wp_p[MODE == BWD_DKV ? 2 : 1];   // BWD_DKV: the weights P (wp holds dS)
      floatx4 pf[2][2];                        // exponents, then P before rounding, then dS
      // BWD_DKV: scalars of the lane's columns, per column tile (a block reads those of the next one in its last slots)
      floatx4 (&l4)[2] = l4_keep;
      floatx4 (&d4)[2] = d4_keep;
      // Pair u = 4 * rt + 2 * ct + h: columns 16 * ct + 4 * g4 + 2 * h, + 1 of row tile rt.  Exponents of P ...
      auto p_fma = [&](int u) {
        const int rt = u >> 2, ct = (u >> 1) & 1, h = u & 1;
#pragma unroll
        for (int e = 2 * h; e < 2 * h + 2; ++e)
          pf[ct][rt][e] = __builtin_fmaf(s_cur[ct][rt][e], c2, -(ROWS_ARE_QUERIES ? L2_row[rt] : l4[ct][e]));
      };
      // ... P (one of the pair), unrounded for dS ...
      auto p_exp = [&](int u, int v) {
        const int rt = u >> 2, ct = (u >> 1) & 1, e = 2 * (u & 1) + v;
        pf[ct][rt][e] = __builtin_amdgcn_exp2f(pf[ct][rt][e]);
      };
      auto pack = [&](bf16x8 (&to)[2], const floatx4 (&from)[2][2], int u) {
        const int rt = u >> 2, ct = (u >> 1) & 1, h = u & 1;
        floatx2 f2 = {from[ct][rt][2 * h], from[ct][rt][2 * h + 1]};
        bf16x2 h2 = __builtin_convertvector(f2, bf16x2);
        to[rt][4 * ct + 2 * h] = h2[0];
        to[rt][4 * ct + 2 * h + 1] = h2[1];
      };
      // ... and dS = P * (dP - D): the accumulators of dP start from -D
      auto ds_mul = [&](int u) {
        const int rt = u >> 2, ct = (u >> 1) & 1, h = u & 1;
#pragma unroll
        for (int e = 2 * h; e < 2 * h + 2; ++e) pf[ct][rt][e] *= dp[ct][rt][e];
      };
      constexpr int NSLOT = 2 * NFRAG;
      // LDS instructions per operand, and those issued behind the request of operand f before its wait (in
      // slot 2 * f - 1): the operands' and the next block's scalars'
      constexpr auto reads_of = [](int f) { return f % NFRAG < 16 ? 1 : 2; };
      constexpr auto scalar_slot = [](int i) { return MODE == BWD_DKV && i >= 50 && i <= 56 && i % 2 == 0; };
      constexpr auto pending = [=](int f) {
        int n = 0;
        for (int x = f + 1; x < f + LA - 1; ++x) n += reads_of(x);
        for (int i = 2 * (f - LA) + 2; i < 2 * f; ++i) n += scalar_slot((i + NSLOT) % NSLOT);
        return n < 15 ? n : 15;
      };
      // slots 26, 30, .. 58 (every 2nd, 4th or 7th from 0, 2, 26 or 42 on: the same within 0.2 %)
      constexpr auto request_at = [](int i) { return i >= 26 && i % 4 == 2 ? (i - 26) / 4 : REQUESTS; };
      static_assert(!REQUEST || request_at(58) == REQUESTS - 1, "every request has its slot");
      // (compile-time slot numbers: a loop of this size is beyond what the compiler unrolls in full)
      static_for<0, NSLOT>([&](auto slot_c) {
        constexpr int i = decltype(slot_c)::value;
        constexpr int f = i >> 1, rt = i & 1;
        const bf16x8 a = fr[f % LA];
        if constexpr (f < 8) dp[f & 1][rt] = mfma(a, r2f[rt][f >> 1], f >= 2 ? dp[f & 1][rt] : MODE == BWD_DKV ? d4[f & 1] : nd_row[rt]);  // from -D
        else if constexpr (f < 16) s_next[f & 1][rt] = mfma(a, r1f[rt][(f - 8) >> 1], f < 10 ? zero4 : s_next[f & 1][rt]);
        else if constexpr (f < 24 && MODE == BWD_DKV) acc_v[f - 16][rt] = mfma(a, wp_p[rt], acc_v[f - 16][rt]);
        else acc[f - (NFRAG - 8)][rt] = mfma(a, wp[rt], acc[f - (NFRAG - 8)][rt]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (rt == 1) {
          __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (pending(f + 1) << 8));  // (LDS reads only)
          fr[f % LA] = fetch(f + LA);
        }
        if constexpr (MODE == BWD_DKV) {  // the next block's scalars, when this block has used its own for the last time
          if (i == 50) l4[0] = *reinterpret_cast<const floatx4*>(scn);
          if (i == 52) l4[1] = *reinterpret_cast<const floatx4*>(scn + 16);
          if (i == 54) d4[0] = *reinterpret_cast<const floatx4*>(scn + 64);
          if (i == 56) d4[1] = *reinterpret_cast<const floatx4*>(scn + 64 + 16);
        }
        if constexpr (REQUEST && request_at(i) < REQUESTS) request_one(ic<request_at(i)>{}, free_slot);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (i >= 1 && i < 25) {
          constexpr int u = (i - 1) / 3, part = (i - 1) % 3;
          if (part == 0) p_fma(u);
          else p_exp(u, part - 1);
        }
        if constexpr (MODE == BWD_DKV) {
          if constexpr (i >= 25 && i < 29) {
            pack(wp_p, pf, 2 * (i - 25));
            pack(wp_p, pf, 2 * (i - 25) + 1);
          }
          if constexpr (i >= 29 && i < 37) ds_mul(i - 29);
          if constexpr (i >= 37 && i < 41) {
            pack(wp, pf, 2 * (i - 37));
            pack(wp, pf, 2 * (i - 37) + 1);
          }
        } else if constexpr (i >= 24 && i < 32) {  // (two wavefronts per SIMD: three in a slot cost nothing)
          ds_mul(i - 24);
          pack(wp, pf, i - 24);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int t4 = 0; t4 < 4; ++t4) s_cur[t4 >> 1][t4 & 1] = s_next[t4 >> 1][t4 & 1];
      have = true;
    });
    advance(cur);
    {
      const int next = slot_after(ring);
      const int d0 = next - ring, d1 = slot_after(next) - next;
      ring = next;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        kb0[i] += d0;
        vb0[i] += d0;
        kb1[i] += d1;
        // (opaque to the compiler, which would otherwise keep the lane parts and add the slot at every read)
        asm volatile("" : "+v"(kb0[i]), "+v"(vb0[i]), "+v"(kb1[i]));
      }
      if (!ROWS_ARE_QUERIES) {
        sb0 += d0;
        sb1 += d1;
        asm volatile("" : "+v"(sb0), "+v"(sb1));
      }
    }
  }
  if (SPREAD) __builtin_amdgcn_s_waitcnt((0 & 15) | (7 << 4) | (15 << 8) | (0 << 14));  // vmcnt(0): the repeated requests

  // ---------------------------------------------------------------- scale, round, store
  if (!wave_active) return;
  if constexpr (ALT) {  // wavefronts 2, 3 hand their sums to 0, 1 through the ring, which nobody reads any more
    static_assert(MODE == BWD_DKV && NW == 4 && 2 * 32 * 64 * 16 <= bwd_ring_slots(MODE) * bwd_slot(MODE), "64 KB");
    floatx4* const hand = reinterpret_cast<floatx4*>(smem) + (wave & 1) * 32 * 64 + lane;
    __syncthreads();
    if (wave >= 2)
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          hand[(2 * dt + rt) * 64] = acc[dt][rt];
          hand[(16 + 2 * dt + rt) * 64] = acc_v[dt][rt];
        }
    __syncthreads();
    if (wave >= 2) return;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        acc[dt][rt] += hand[(2 * dt + rt) * 64];
        acc_v[dt][rt] += hand[(16 + 2 * dt + rt) * 64];
      }
  }
  // (What the results' stores need is read from the kernel arguments here, not carried through the
  // main loop in scalar registers, which it has too few of.)
  typedef const __attribute__((address_space(4))) BParams* ArgsPtr;
  ArgsPtr ka = (ArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(ka));
  if (PARTIAL && RMAP::num_sets(p.geom) > 1) {
    // fp32 partial sums: part[((set * B + batch) * Hkv + kvh) * keys + row][128] of dk, behind all of them those of dv
    int keys = n_rows;
    if constexpr (ALT) keys = map.ns;
    const int64_t all = (int64_t)RMAP::num_sets(p.geom) * nbh * keys * 128;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
      if (row_valid[rt]) {
        float* prow = ka->part + ((((int64_t)set * ka->B + batch) * ka->Hkv + kvh) * keys + row[rt]) * 128 + 4 * g4;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
          *reinterpret_cast<floatx4*>(prow + 16 * dt) = acc[dt][rt] * ka->scale;
          *reinterpret_cast<floatx4*>(prow + all + 16 * dt) = acc_v[MODE == BWD_DKV ? dt : 0][rt];
        }
      }
    return;
  }
  // The four lanes of a row hold head dims 4 * g4 .. + 3 of every 16-dim tile; a lane quarter and
  // its neighbour trade 8 bytes per tile pair so that each lane owns the whole 16-byte chunk
  // 4 * m + 2 * (g4 % 2) + g4 / 2 of its row.
  enum { TO_DQ, TO_DK, TO_DV };
  auto store_rows = [&](const floatx4 (&a)[8][2], int what, float factor) {
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const bool keep = row_valid[rt] && map.store((int)rpos[rt]);
      uint16_t* orow;
      if (what == TO_DQ) orow = ka->dq + (batch * ka->dq_bs + rpos[rt] * ka->dq_rs + hq * ka->dq_hs + chunk_ofs);
      else if (what == TO_DK) orow = ka->dk + (batch * ka->dk_bs + rpos[rt] * ka->dk_rs + kvh * ka->dk_hs + chunk_ofs);
      else orow = ka->dv + (batch * ka->dv_bs + rpos[rt] * ka->dv_rs + kvh * ka->dv_hs + chunk_ofs);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        uint32_t w[2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int k2 = 0; k2 < 2; ++k2) {
            floatx2 v2 = {a[2 * m + t][rt][2 * k2] * factor, a[2 * m + t][rt][2 * k2 + 1] * factor};
            w[t][k2] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2, bf16x2));
          }
        auto q0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
        auto q1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
        if (keep) {
          u32x4 pk = {q0[0], q1[0], q0[1], q1[1]};
          if constexpr (RMAP::kAccumulate) {  // add to what an earlier pass has written (both rounded to bf16)
            const u32x4 old = what == TO_DK ? old_k[rt][m] : old_v[rt][m];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              floatx2 s2 = {__uint_as_float(pk[i] << 16) + __uint_as_float(old[i] << 16),
                            __uint_as_float(pk[i] & 0xffff0000u) + __uint_as_float(old[i] & 0xffff0000u)};
              pk[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(s2, bf16x2));
            }
          }
          *reinterpret_cast<u32x4*>(orow + 32 * m) = pk;
        }
      }
    }
  };
  if constexpr (MODE == BWD_DKV) {
    store_rows(acc, TO_DK, ka->scale);
    store_rows(acc_v, TO_DV, 1.f);
  } else {
    store_rows(acc, TO_DQ, ka->scale);
  }
}

struct NoLeadingKeys {};

// One launch: the workgroups of RMAP and, with LEAD, those of a second kind of rows - for dK / dV the keys
// that every (later) query sees (KeyRowsLeading), for dQ of image Gather 0 the text queries (below).  The leading keys are few rows with very many columns, whose launch of its own
// had one thin round of workgroups; here the rest of the GPU works on the other keys meanwhile.  The
// longer kind of workgroup comes first, so that the short ones fill the last round.  Against two
// launches of their own, dK (three products) and dV (two) with 8 wavefronts: a training step with 64
// sinks 551 -> 505 us (window 575, S = 8192, 32 / 8 heads), 870 -> 817 us (block Scatter G = 2,
// S = 6000), image Scatter 1024^2 at 24 heads 339 -> 327 us.
// dQ of image Gather 0: the text rows and the patch runs have maps of their own.  One map for both
// chose between their fields at every tile (383 scalar instructions per step of two blocks, 46 of
// them and 2 more moving spilled scalars; the patch runs alone issue 291 and 18).
// With that and shared row blocks for the text rows, 1024^2 at 24 heads: the launch 115 -> 90 us (two
// traces), the training step 345 -> 323.
template <class RMAP, int MODE, int HP, class LEAD, bool FAR>
__global__ __launch_bounds__(bwd_waves(MODE) * 64, MODE == BWD_DKV ? 1 : 2) void intra_bwd_kernel(const BParams p) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[bwd_ring_slots(MODE) * bwd_slot(MODE)];
  int block = blockIdx.x;
  if constexpr (!std::is_same_v<LEAD, NoLeadingKeys>) {
    const int lead_block = block - (p.lead_first ? 0 : p.grid.blocks);
    if (lead_block >= 0 && lead_block < p.lead.blocks) {
      bwd_rows<LEAD, MODE, HP, MODE == BWD_DKV, FAR>(p, p.lead, lead_block, smem);
      return;
    }
    if (p.lead_first) block -= p.lead.blocks;
  }
  bwd_rows<RMAP, MODE, HP, false, FAR>(p, p.grid, block, smem);
}

// Adds up the partial sums of the leading keys over the chunks and writes their rows of dk
// (blockIdx.y == 0) or dv: one thread per (batch, kv head, key, 4 head dims).  Eight chunks are
// requested before the first is added: a chain of one load per chunk is latency only.
__global__ void intra_bwd_lead_reduce(const BParams p, int n_chunks, int ns) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t rows = (int64_t)p.B * p.Hkv * ns;
  if (i >= rows * 32) return;
  const int d4 = (int)(i & 31);
  const int64_t row = i >> 5;  // (batch * Hkv + kvh) * ns + key
  const float* part = p.part + ((blockIdx.y ? n_chunks * rows : 0) + row) * 128 + 4 * d4;
  floatx4 s = {0.f, 0.f, 0.f, 0.f};
  int c = 0;
  for (; c + 8 <= n_chunks; c += 8) {
    floatx4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = *reinterpret_cast<const floatx4*>(part + (c + k) * rows * 128);
#pragma unroll
    for (int k = 0; k < 8; ++k) s += v[k];
  }
  for (; c < n_chunks; ++c) s += *reinterpret_cast<const floatx4*>(part + c * rows * 128);
  const int key = (int)(row % ns);
  const int64_t bh = row / ns;
  const int kvh = (int)(bh % p.Hkv), batch = (int)(bh / p.Hkv);
  floatx2 a = {s[0], s[1]}, b = {s[2], s[3]};
  uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(a, bf16x2));
  uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(b, bf16x2));
  uint16_t* o = blockIdx.y ? p.dv + (batch * p.dv_bs + key * p.dv_rs + kvh * p.dv_hs + 4 * d4)
                           : p.dk + (batch * p.dk_bs + key * p.dk_rs + kvh * p.dk_hs + 4 * d4);
  *reinterpret_cast<uint2*>(o) = make_uint2(lo, hi);
}

}  // namespace intra
