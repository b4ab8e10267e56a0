// Host-side launch plan of the block-selection kernels: validated dimensions, work-unit sizes
// and the byte layout of the three caller-owned workspaces.  Recomputed from the descriptor on
// every call (pure function, a few dozen integer operations), passed to kernels by value.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include "../../include/nsa_hip.h"

#ifndef NSA_PHASE_BYTES
#define NSA_PHASE_BYTES (1L << 22)
#endif

#ifndef NSA_DKV_UNITS_WANTED
#define NSA_DKV_UNITS_WANTED 4096
#endif
#ifndef NSA_DKV_CHUNK_FIXED
#define NSA_DKV_CHUNK_FIXED 0      // a power of two to override the choice (experiments)
#endif

namespace nsa {

struct SelPlan {
  int b, hkv, g, lg, n, S, SP, B, D, causal, W, nch, bh, idx64;
  float scale;
  // Work-unit tables.  A unit = up to `chunk` consecutive pairs of one (query phase, block)
  // cell; cells are ordered phase-major so that units running at the same time gather Q rows of
  // the same query range (L2 reuse).  Table t: 0 = forward walk, 1 = dQ walk, 2 = dK/dV walk
  // (a single phase: the whole sequence, so a wave keeps its dK/dV accumulators as long as
  // possible), 3 = the same for sel_bwd_dkv_kernel where sel_bwd_block_kernel reads table 2.
  int tables;                // 3, or 4 where both dK/dV walks may run: which of them does, each backward call decides
  int chunk[4], phase[4], np[4], ub[4];
  size_t off_unit[4];
  size_t off_urec[4];        // per (batch*kv head, unit) a record of 8 ints: block, own, list start, v0, v1
  int ub_kv;                 // dK/dV partials reserved per (batch, kv head): the longer of the tables
  long list_cap;             // inverse-index entries reserved per (batch, kv head)
  size_t prow;               // number of partial rows; padding rows write to the spare rows behind them: one in the forward, g in the backward
  long sq[3], sk[3], sv[3], so[3];
  // index workspace
  size_t off_cnt, off_blk, off_list, index_total;
  // forward workspace
  size_t off_opart, off_lsepart, fwd_total;
  // backward workspace
  size_t off_delta, off_dqpart, off_dkvpart, off_ticket, bwd_total;
  int near_rows;             // byte offsets of a kv head's Q rows fit 32 bits
  int block_walk;            // the backward walk without gate gradients is sel_bwd_block_kernel
};

// x / d for x < 2^31 (Granlund and Montgomery 1994): high word of 2 x * mul, shifted right by sh
struct SmallDiv {
  unsigned mul;
  int sh;
};
static inline SmallDiv small_div(int d) {
  int l = 0;
  while ((1 << l) < d) ++l;
  return {(unsigned)((((unsigned long)1 << (31 + l)) + d - 1) / d), l};
}

static inline size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

static inline int make_plan(const nsa_select_desc* d, SelPlan& P) {
  if (!d) return NSA_E_ARG;
  if (d->batch <= 0 || d->kv_heads <= 0 || d->group <= 0 || d->seq <= 0 || d->num_sel < 0 || d->block <= 0) return NSA_E_ARG;
  if (d->dim_head != 64 && d->dim_head != 128) return NSA_E_UNSUPPORTED;
  if (d->block > 64) return NSA_E_UNSUPPORTED;                 // a block is one or two 32-key register tiles; keys past the block are masked
  if (d->group > 32 || (d->group & (d->group - 1))) return NSA_E_UNSUPPORTED;
  if (d->num_sel > 62) return NSA_E_UNSUPPORTED;
  if (!d->causal && d->num_sel == 0) return NSA_E_ARG;
  P.b = d->batch; P.hkv = d->kv_heads; P.g = d->group; P.n = d->seq; P.S = d->num_sel; P.SP = d->num_sel + 1;
  P.B = d->block; P.D = d->dim_head; P.causal = d->causal ? 1 : 0; P.idx64 = d->idx_is_int64 ? 1 : 0;
  P.scale = d->scale;
  P.lg = 0;
  while ((1 << P.lg) < P.g) ++P.lg;
  P.W = (P.n + P.B - 1) / P.B;
  if (P.W > 16384) return NSA_E_UNSUPPORTED;
  if ((long)P.n * P.SP >= 0x7fffffffL) return NSA_E_UNSUPPORTED;
  P.nch = (P.n + 255) / 256;
  const long bh = (long)P.b * P.hkv;
  if (bh > 65535) return NSA_E_UNSUPPORTED;
  P.bh = (int)bh;
  for (int t = 0; t < 3; ++t) { P.sq[t] = d->q_stride[t]; P.sk[t] = d->k_stride[t]; P.sv[t] = d->v_stride[t]; P.so[t] = d->o_stride[t]; }
  for (int t = 0; t < 3; ++t)
    if ((P.sq[t] | P.sk[t] | P.sv[t] | P.so[t]) & 7) return NSA_E_ARG;      // rows must start 16-byte aligned
  for (int t = 1; t < 3; ++t)                                               // head and token strides: 32-bit arithmetic in the gathers
    if ((P.sq[t] | P.so[t]) < 0 || ((P.sq[t] | P.so[t]) >> 32)) return NSA_E_UNSUPPORTED;
  const long pairs = (long)P.n * (P.S + P.causal);
  // phase length: the Q rows (forward) / Q and dO rows (dQ walk) of one phase are about the size
  // of one XCD's 4 MB L2 (measured best on MI355X among 0.5 .. 64 MB; shorter phases make the
  // work units too small, longer ones lose the L2 reuse of the gathered rows)
  const long row_bytes = (long)P.g * P.D * 2;
  long ph = 256;
  while (ph * 2 * row_bytes <= (long)NSA_PHASE_BYTES && ph < (1L << 20)) ph *= 2;
  // A unit is a serial chain of its pairs, 32 / group of them at a time, and a short sequence has few blocks: 289 tokens of 2 kv heads
  // were 30 units of 256 pairs on 1024 SIMDs.  Shorter units where the launch would have under 2048 (a pair's results do not depend on
  // its unit).  us with index build and merge, 256 pairs / this rule: 289 tokens, 16 / 2 heads, d 128, 15 blocks of 64 128 / 44; 1 x 512,
  // 8 / 2 heads, 4 of 16 50 / 30; 2000, 16 / 2, d 128 160 / 99; 4 x 1024, 16 / 4 107 / 85; 4096, 16 / 4 116 / 98.  At 4096 units the last two
  // take 85 and 103, 2 x 687 with 32 / 8 heads 99 instead of 92, 1 x 4000 of d 128 260 instead of 250.
  long per = 256;
  while (per > 32 && bh * pairs / per < 2048) per /= 2;
  P.chunk[0] = (int)per;  P.phase[0] = (int)ph;
  P.chunk[1] = (int)per;  P.phase[1] = (int)(ph > 256 ? ph / 2 : ph);
  // dK/dV walk: a unit keeps its accumulators for `chunk` pairs and leaves a 2 x 32KT x D fp32 partial behind, so long units
  // are cheaper per pair - but the chip holds 512 to 1024 work-groups of this kernel at a time, and a launch with fewer
  // units than a few rounds of that runs as long as its longest units whatever the rest does (seq 8k, 4 kv heads: 512 units
  // of 1024 pairs occupy half of the SIMDs for the whole launch).  Shorter units when the launch would have under ~4096.
  // (shapes whose backward walk is sel_bwd_block_kernel where the strides allow it.  With fewer heads a group its row gathers have an
  // offset per lane: 4096 tokens of 8 / 8 heads 150 us against the two-wave walk's 120, of 8 / 4 heads 109 against 98)
  const bool long_units = P.D == 128 && P.B > 32 && P.g >= 4;
  P.tables = long_units ? 4 : 3;
  P.chunk[3] = 0;
  {
    const long want = bh * pairs / NSA_DKV_UNITS_WANTED;
    P.chunk[2] = NSA_DKV_CHUNK_FIXED ? NSA_DKV_CHUNK_FIXED : (want >= 1024 ? 1024 : want >= 512 ? 512 : 256);
    // ... down to 64 pairs while there are under 512 of them: 289 tokens of 16 / 2 heads, d 128 138 / 62 us, 1 x 512 of 8 / 2 49 / 28 and of
    // d 128 81 / 54, 1200 of 16 / 2, d 128 154 / 107 (units of 32 pairs: 59, 24, 66, 146; under 1024: 1899 of 16 / 4 83 instead of 71)
    while (P.chunk[2] > 64 && bh * pairs / P.chunk[2] < 512) P.chunk[2] /= 2;
    // sel_bwd_block_kernel takes a unit with four waves on one of 256 work-groups: few long units, about four for each of them while a
    // unit is long, one for each below.  us of walk + reduction, 32 / 8 heads, 15 blocks, units of 256 / 512 / 1024 / 2048 pairs: 2048
    // tokens 155 / 150 / 148, 4096 313 / 273 / 294 / 291, 8192 648 / 550 / 528 / 579, 32768 2630 / 2209 / 2010 / 1987; 16 / 2 heads, 64 / 128 /
    // 256 / 512 pairs: 289 tokens 46 / 51 / 65 / 69, 1200 98 / 71 / 77 / 110, 2000 163 / 116 / 91 / 117
    if (long_units && !NSA_DKV_CHUNK_FIXED) {
      P.chunk[2] = 2048;
      while (P.chunk[2] > 512 && bh * pairs / P.chunk[2] < 1000) P.chunk[2] /= 2;
      while (P.chunk[2] > 64 && bh * pairs / P.chunk[2] < 250) P.chunk[2] /= 2;
      // The two-wave walk at these shapes (gate gradients, far strides) has 512 work-groups on the chip and wants twice the units while they
      // are short of 1024 pairs; slots beyond the number of blocks are dead.  us of a backward with gate gradients, units of 64 / 128 / 256 /
      // 512 / 1024 / 2048 pairs: 16 / 2 heads, 15 blocks: 1000 tokens 129 / 125, 2000 218 / - / 203, 3000 300 / 267 / 245, 4096 383 / 324 /
      // 331 / 360, 8192 822 / 649 / 667 / 706; 32 / 8 heads, 16 blocks: 400 tokens 70 / 72, 1024 180 / 157 / 141 / 177, 2048 - / 307 / 277 / 291,
      // 4096 - / 681 / 620 / 588 / 625, 8192 - / - / 1286 / 1237 / 1234 / 1377, 16384 - / - / 2571 / 2455 / 2470 / 2545, 32768 - / - / 5150 /
      // 4905 / 4937 / 4820
      const long live = bh * P.n * ((P.S < P.W ? P.S : P.W) + P.causal);
      P.chunk[3] = live / 2048 >= 2000 ? 2048 : 1024;
      while (P.chunk[3] > 256 && live / P.chunk[3] < 1000) P.chunk[3] /= 2;
      while (P.chunk[3] > 64 && live / P.chunk[3] < 250) P.chunk[3] /= 2;
    } else if (long_units) {
      P.chunk[3] = P.chunk[2];
    }
  }
  P.phase[2] = P.phase[3] = ((P.n + 255) / 256) * 256;
  P.np[3] = P.ub[3] = 0;
  for (int t = 0; t < P.tables; ++t) {
    P.np[t] = (P.n + P.phase[t] - 1) / P.phase[t];
    const long cells = (long)P.np[t] * P.W;
    const long ub = cells + (pairs + P.chunk[t] - 1) / P.chunk[t];
    if (ub > 0x3fffffffL) return NSA_E_UNSUPPORTED;
    P.ub[t] = (int)ub;
  }
  P.ub_kv = P.ub[2] > P.ub[3] ? P.ub[2] : P.ub[3];
  P.list_cap = (long)P.n * (P.S > 0 ? P.S : 1);

  size_t o = 0;
  P.off_cnt = o;    o = align_up(o + (size_t)bh * P.nch * P.W * 4);
  P.off_blk = o;    o = align_up(o + (size_t)bh * (P.W + 1) * 4);
  for (int t = 0; t < P.tables; ++t) { P.off_unit[t] = o; o = align_up(o + (size_t)bh * ((size_t)P.np[t] * P.W + 1) * 4); }
  for (int t = 0; t < P.tables; ++t) { P.off_urec[t] = o; o = align_up(o + (size_t)bh * (size_t)P.ub[t] * 32); }
  P.off_list = o;   o = align_up(o + (size_t)bh * P.list_cap * 4);
  P.index_total = o;

  const size_t prow = (size_t)bh * P.n * P.SP * P.g;      // partial rows: (query, slot, head)
  P.prow = prow;
  o = 0;
  P.off_opart = o;   o = align_up(o + (prow + 1) * P.D * 2);
  P.off_lsepart = o; o = align_up(o + (prow + 1) * 4);
  P.fwd_total = o;

  // sel_bwd_block_kernel addresses a kv head's Q and d_out rows, a block's K and V rows and the pairs of all heads with 32 bits
  const long far_q = 2 * ((P.n - 1) * P.sq[2] + (P.g - 1) * P.sq[1] + P.D), far_o = 2 * ((P.n - 1) * P.so[2] + (P.g - 1) * P.so[1] + P.D);
  P.near_rows = far_q <= 0xffffffffL;
  P.block_walk = long_units && P.near_rows && far_o <= 0xffffffffL && P.sk[2] >= 0 && P.sk[2] < (1L << 24) && P.sv[2] >= 0 && P.sv[2] < (1L << 24) &&
                 bh * P.n * P.SP <= 0xffffffffL && P.scale > 0.f;      // (masked scores are -inf before they are scaled)
  const int KT = (P.B + 31) / 32;
  o = 0;
  P.off_delta = o;   o = align_up(o + (size_t)bh * P.g * P.n * (long_units ? 8 : 4));
  P.off_dqpart = o;  o = align_up(o + (prow + P.g) * P.D * 2);
  P.off_dkvpart = o; o = align_up(o + (size_t)bh * P.ub_kv * 2 * 32 * KT * P.D * 4);
  P.off_ticket = o;  o = align_up(o + 4);
  P.bwd_total = o;
  return 0;
}

}  // namespace nsa
