// Single-token decode attention over the key / value caches (NSA.py:338-547): the G query
// heads of one kv head attend either to a contiguous key range (compressed branch, with the
// memory slots as extra keys and the scaled logits written out for the importance scores;
// sliding branch) or to the selected blocks plus the query's own block (selection branch).
//
// HBM-bound: every cached key / value row a query attends is read once.  The keys of a unit
// (batch, kv head) are cut into 32-key tiles that are dealt round-robin to the waves of
// `nsplit` work-groups (split-K), so that a single long sequence still fills the chip; every
// wave keeps a running (max, sum, O) and writes one fp32 partial, and a second kernel merges the
// partials of a head.  Rows are fetched one tile ahead with whole-row coalesced loads and become
// MFMA operands through a per-wave LDS tile (row operand for K, transposing LDS load for V^T):
// reading each row in 32-byte pieces straight into the operand layout touches every cache line
// from several instructions and re-fetches it from L2 once the L1 thrashes.  Scores are computed transposed, S^T = K Q^T on the 32x32x16 MFMA with the
// query heads as (zero-padded) columns: a lane then owns one head, the softmax statistics are
// per-lane scalars and the rescaling of O^T = V^T P needs no cross-lane traffic.
#include "nsa_common.hpp"
#include "../../include/nsa_hip.h"

namespace nsa {

struct DecodePlan {
  int b, hk, g, d;
  int units;         // per batch: hk (shared selection / ranges) or hk*g (per-head selection)
  int gc;            // query heads per unit
  int mode, start, count, mem;
  int B, S, kv_len, tps;
  int tiles, nsplit, nparts, rec;    // rec: floats per partial record: [gc][d] O, [gc] max, [gc] sum, padded to 16 bytes
  int idx64;
  float scale;
  long sq[2], sk[3], sv[3];
  int sstride, lstride;              // row strides of the selection (idx / fmask) and of the logits output
  // Lengths read at run time, for a step replayed from a captured graph: dyn[0] = rows in the key / value caches before
  // this token, dyn[1] = compressed keys cached.  The fields above then hold capacities (the grid and the partial
  // records are sized for them) and resolve() replaces them inside the kernel.
  const int* dyn;
  int dyn_kind;                      // 1 compressed range, 2 selected blocks, 3 sliding window
  int window, per_block, smax;
  int cap_len, cap_nc;               // rows the key / value caches and the compressed caches hold: the counters are clamped to them
};

__device__ __forceinline__ void resolve(DecodePlan& P) {
  if (P.dyn == nullptr) return;
  // a caller that replays the step more often than the caches have rows must not make the kernels read or write past them
  const int kv_len = min(max(P.dyn[0], 0) + 1, P.cap_len), nc = min(max(P.dyn[1], 0), P.cap_nc);
  if (P.dyn_kind == 1) {
    P.count = nc;
    if (nc == 0) P.mem = 0;                            // no compressed key yet: the branch contributes nothing (NSA.py:401)
    P.tiles = ((P.mem + 31) >> 5) + ((nc + 31) >> 5);
  } else if (P.dyn_kind == 2) {
    P.kv_len = kv_len;
    P.S = min(P.smax, nc / P.per_block);
    P.tiles = (P.S + 1) * P.tps;
  } else {
    const int w = min(kv_len, P.window + 1);
    P.start = kv_len - w;
    P.count = w;
    P.tiles = (w + 31) >> 5;
  }
}

constexpr int kDecodeWaves = 2;      // waves per work-group; each stages its own K / V tile in LDS

struct DecodeTile {
  const __bf16 *kb, *vb;             // row 0 of the tile
  long ks, vs;                       // row strides
  int nvalid, lcol;                  // rows in use; column of row 0 in the logits row (-1: not written)
};

// tile t of unit (b, hk, ug) -> its rows; nvalid <= 0 for tiles with nothing to attend
__device__ __forceinline__ DecodeTile decode_tile(const DecodePlan& P, int D, int t, int b, int hk, int ug, const __bf16* k, const __bf16* v,
                                                  const __bf16* mem_k, const __bf16* mem_v, const void* idx, const unsigned char* fmask, const int* sel_s) {
  DecodeTile T;
  T.lcol = -1;
  if (P.mode == 0) {
    const int mem_tiles = (P.mem + 31) >> 5;
    if (t < mem_tiles) {
      T.kb = mem_k + ((long)hk * P.mem + 32 * t) * D;
      T.vb = mem_v + ((long)hk * P.mem + 32 * t) * D;
      T.ks = T.vs = D;
      T.nvalid = min(32, P.mem - 32 * t);
    } else {
      const int tt = t - mem_tiles;
      T.kb = k + b * P.sk[0] + hk * P.sk[1] + (long)(P.start + 32 * tt) * P.sk[2];
      T.vb = v + b * P.sv[0] + hk * P.sv[1] + (long)(P.start + 32 * tt) * P.sv[2];
      T.ks = P.sk[2]; T.vs = P.sv[2];
      T.nvalid = min(32, P.count - 32 * tt);
      T.lcol = 32 * tt;
    }
  } else {
    const int slot = t / P.tps, sub = t % P.tps;
    long blk;
    bool live = true;
    if (slot < P.S && sel_s != nullptr) {             // selected by this work-group: -1 for a dead slot
      blk = sel_s[slot];
      live = (blk >= 0) & (blk * P.B < P.kv_len);
      if (!live) blk = 0;
    } else if (slot < P.S) {
      const long e = (long)ug * P.sstride + slot;
      const unsigned char fm = fmask[e];              // requested together with the index: one round trip, not two
      blk = P.idx64 ? reinterpret_cast<const long*>(idx)[e] : (long)reinterpret_cast<const int*>(idx)[e];
      live = (fm != 0) & (blk >= 0) & (blk * P.B < P.kv_len);
      if (!live) blk = 0;
    } else {
      blk = (P.kv_len - 1) / P.B;                     // the query's own block, up to itself
    }
    const long key0 = blk * P.B + 32 * sub;
    T.kb = k + b * P.sk[0] + hk * P.sk[1] + key0 * P.sk[2];
    T.vb = v + b * P.sv[0] + hk * P.sv[1] + key0 * P.sv[2];
    T.ks = P.sk[2]; T.vs = P.sv[2];
    T.nvalid = live ? (int)min((long)32, min((long)P.B - 32 * sub, (long)P.kv_len - key0)) : 0;
  }
  return T;
}

// What a work-group does beside attending its keys (a whole decode step is then three launches: compressed keys + window,
// selected blocks, merge - a launch that depends on another costs 4-5 us, as much as these kernels themselves at batch 1):
//   kPooled    compressed keys: leaves the importance logits pooled per selection block instead of one per key and head
//   kNewToken  sliding window: rotates the queries, takes the newest key / value from the projection and puts both into the caches
//   kTopk      selected blocks: selects them itself from the pooled logits
enum { kPlain = 0, kPooled = 1, kNewToken = 2, kTopk = 3 };

struct PoolOut {                     // kPooled: fp32 [batch, units, stride]; one row per kv head (share) or per query head
  float* out;
  long stride;
  int npf, share;                    // compressed keys per block (1, 2, 4 .. 32); the group's heads share a row
};
struct NewToken {                    // kNewToken
  const __bf16 *k, *v;               // projections, un-rotated, element strides {batch, head}
  long k0, k1, v0, v1;
  const void* freqs;                 // fp32, or bf16 when freqs_bf16
  int freqs_bf16;
  __bf16* rq;                        // rotated queries [batch, heads, D] for the selected-block branch
  __bf16 *kc, *vc;                   // the caches (strides as in the plan)
  __bf16 *krun, *vrun;               // open compression window (optional): row address, or a ring when ring > 0
  long ku0, ku1, vu0, vu1, ku_row, vu_row;
  int ring;
};
struct TopkIn {                      // kTopk
  const float* pooled;
  long stride;
  int nb, per_block, kstride;        // blocks in a row (run-time count: dyn[1] / per_block), row stride of the results
  int* idx;
  unsigned char* fm;
};

// One branch of a decode step: what a launch needs besides the grid.
struct AttendArgs {
  DecodePlan P;
  const __bf16 *q, *k, *v, *mem_k, *mem_v;
  const void* idx;
  const unsigned char* fmask;
  float* part;
  float* logits;
  PoolOut pool;
  NewToken nt;
  TopkIn topk;
};

__device__ __forceinline__ float wave_reduce_max(float v) {
#pragma unroll
  for (int o = 1; o <= 32; o <<= 1) v = fmaxf(v, o == 1 ? dpp_quad_xor1(v) : o == 2 ? dpp_quad_xor2(v) : __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_reduce_sum(float v) {
#pragma unroll
  for (int o = 1; o <= 32; o <<= 1) v += o == 1 ? dpp_quad_xor1(v) : o == 2 ? dpp_quad_xor2(v) : __shfl_xor(v, o, 64);
  return v;
}

// Block selection of one row by one wave (NSA.py:693-713, 721: softmax with the extra -1e3 column, the k largest in descending
// order, equal ones lower index first; a slot is live when its probability exceeds 1e-10).  nb <= 2048, k <= min(64, nb).
// Lane l holds entries l, l + 64, ...  The k-th largest of the 64 lanes' maxima (a bitwise search with ballots: 31 steps) is a
// lower bound of the k-th largest entry that only a few entries beyond the k reach; those are listed in LDS, a lane takes
// one and counts the listed ones that come before it: its slot.  (Extracting maxima one by one, k dependent rounds of a wave
// maximum and a re-scan: 16 us for 8 rows of 512 with k = 16.)  sel[slot] = block, or -1 for a dead slot.
__device__ __forceinline__ void wave_topk(const float* __restrict__ row, int nb, int k, int lane, float* __restrict__ cand_p, int* __restrict__ cand_j,
                                          int* __restrict__ sel, int* __restrict__ idx_out, unsigned char* __restrict__ fm_out) {
  const int vpl = (nb + 63) >> 6;
  float x[32];
  float mx = -1e3f;
#pragma unroll
  for (int c = 0; c < 32; c += 8) {
    if (c >= vpl) continue;                               // wave-uniform
#pragma unroll
    for (int r = c; r < c + 8; ++r) x[r] = r * 64 + lane < nb ? row[r * 64 + lane] : -INFINITY;
  }
#pragma unroll
  for (int c = 0; c < 32; c += 8) {
    if (c >= vpl) continue;
#pragma unroll
    for (int r = c; r < c + 8; ++r) mx = fmaxf(mx, x[r]);
  }
  mx = wave_reduce_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < 32; c += 8) {
    if (c >= vpl) continue;
#pragma unroll
    for (int r = c; r < c + 8; ++r) { x[r] = __expf(x[r] - mx); sum += x[r]; }
  }
  sum = wave_reduce_sum(sum) + __expf(-1e3f - mx);
  const float inv = 1.0f / sum;
  int top = 0;                                             // probabilities as integers: same order, padding negative
#pragma unroll
  for (int c = 0; c < 32; c += 8) {
    if (c >= vpl) continue;
#pragma unroll
    for (int r = c; r < c + 8; ++r) {
      float p = x[r] * inv;
      p = (p == p) ? p : INFINITY;                         // NaN (a diverged row): ordered first, like torch.topk
      p = r * 64 + lane < nb ? p : -1.0f;
      x[r] = p;
      top = max(top, __builtin_bit_cast(int, p));
    }
  }
  int T = 0;
  for (int bit = 30; bit >= 0; --bit) {
    const int c = T | (1 << bit);
    if ((int)__popcll(__ballot(top >= c)) >= k) T = c;
  }
  auto count = [&](int v) {                                // entries >= v
    int n = 0;
#pragma unroll
    for (int c = 0; c < 32; c += 8) {
      if (c >= vpl) continue;
#pragma unroll
      for (int r = c; r < c + 8; ++r) n += (int)__popcll(__ballot(__builtin_bit_cast(int, x[r]) >= v));
    }
    return n;
  };
  int ties = 64;                                           // entries equal to T that are listed
  if (count(T) > 64) {                                     // (many equal entries, or the k largest in few lanes: the exact k-th largest)
    T = 0;
    for (int bit = 30; bit >= 0; --bit) {
      const int c = T | (1 << bit);
      if (count(c) >= k) T = c;
    }
    ties = k - count(T + 1);
  }
  int listed = 0;
  const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
  for (int c = 0; c < 32; c += 8) {
    if (c >= vpl) continue;
#pragma unroll
    for (int r = c; r < c + 8; ++r) {
      const int v = __builtin_bit_cast(int, x[r]);
      const unsigned long long eq = __ballot(v == T);
      const bool keep = v > T || (v == T && (int)__popcll(eq & below) < ties);
      const unsigned long long kept = __ballot(keep);
      const int at = listed + (int)__popcll(kept & below);
      if (keep && at < 64) { cand_p[at] = x[r]; cand_j[at] = r * 64 + lane; }
      listed += (int)__popcll(kept);
      ties -= (int)__popcll(eq);
    }
  }
  __builtin_amdgcn_wave_barrier();                         // LDS operations of one wave execute in order
  listed = min(listed, 64);
  const float p = lane < listed ? cand_p[lane] : -1.0f;
  const int j = lane < listed ? cand_j[lane] : 0;
  int rank = 0;
  for (int i = 0; i < listed; ++i) {
    const float pi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), i));
    rank += (pi > p) | ((pi == p) & (i < lane));           // the list is in index order
  }
  if (lane < listed && rank < k) {
    const bool live = p < INFINITY && p > 1e-10f;
    sel[rank] = live ? j : -1;
    if (idx_out != nullptr) { idx_out[rank] = j; fm_out[rank] = live ? 1 : 0; }
  }
}

// Pooled importance logits of one 32-key tile (NSA.py:448-476: mean over a block's npf keys and, if shared, the group's heads):
// key 8 (i / 4) + 4 h + i % 4 of the tile is register i, head n_ the lane.
__device__ __forceinline__ void pool_tile(const DecodePlan& P, const PoolOut& O, const floatx16& S, int lcol, long row, int n_, int h) {
  const float norm = P.scale / (float)(O.npf * (O.share ? P.gc : 1));
  const bool writer = O.share ? n_ == 0 : n_ < P.gc;
  float* dst = O.out + row * O.stride;
  auto put = [&](float v, int key) {                       // block of keys key .. key + npf - 1
    if (O.share)
      for (int o = 1; o < P.gc; o <<= 1) v += o == 1 ? dpp_quad_xor1(v) : o == 2 ? dpp_quad_xor2(v) : __shfl_xor(v, o, 64);      // (lanes past the group hold zeros)
    if (writer && key + O.npf <= P.count) dst[key / O.npf] = v * norm;
  };
  if (O.npf <= 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int key = lcol + 8 * u + 4 * h;
      if (O.npf == 4) put((S[4 * u] + S[4 * u + 1]) + (S[4 * u + 2] + S[4 * u + 3]), key);
      else if (O.npf == 2) { put(S[4 * u] + S[4 * u + 1], key); put(S[4 * u + 2] + S[4 * u + 3], key + 2); }
      else {
#pragma unroll
        for (int e = 0; e < 4; ++e) put(S[4 * u + e], key + e);
      }
    }
  } else {
    float s8[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) s8[u] = halves_sum((S[4 * u] + S[4 * u + 1]) + (S[4 * u + 2] + S[4 * u + 3]));
    if (O.npf == 8) {
#pragma unroll
      for (int u = 0; u < 4; ++u) put(s8[u], lcol + 8 * u);
    } else if (O.npf == 16) { put(s8[0] + s8[1], lcol); put(s8[2] + s8[3], lcol + 16); }
    else put((s8[0] + s8[1]) + (s8[2] + s8[3]), lcol);
  }
}

template <int D>
struct DecodeShared {                // of one work-group, declared once per kernel
  static constexpr int RS = D + 8, RSV = D + 16;      // row reads want 4 banks per row, transpose loads 8
  __align__(16) __bf16 kv[kDecodeWaves][2][32 * RSV];
  float step[2][64];                 // kNewToken: cos / sin of the new position; kTopk: the selection's candidates
  int sel[64];                       // kTopk: the selected blocks
};

// Work-group (bx, blockIdx.y) of a branch: bx = index among the branch's split-K work-groups.
template <int D, int ROLE>
__device__ __forceinline__ void decode_attend_body(const AttendArgs& A, const int bx, DecodeShared<D>& sh) {
  constexpr int KS = D / 16, DT = D / 32, RS = DecodeShared<D>::RS, RSV = DecodeShared<D>::RSV;
  constexpr int LPR = D / 8, RPI = 64 / LPR, NI = 32 / RPI;      // lanes per row, rows per load instruction, instructions per tile
  DecodePlan P = A.P;
  resolve(P);
  const __bf16* __restrict__ q = A.q;
  const __bf16* __restrict__ k = A.k;
  const __bf16* __restrict__ v = A.v;
  const __bf16* __restrict__ mem_k = A.mem_k;
  const __bf16* __restrict__ mem_v = A.mem_v;
  const void* __restrict__ idx = A.idx;
  const unsigned char* __restrict__ fmask = A.fmask;
  float* __restrict__ part = A.part;
  float* __restrict__ logits = A.logits;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n_ = lane & 31, h = lane >> 5;
  const int lr = lane / LPR, lc = lane % LPR;
  __bf16* k_s = sh.kv[wave][0];
  __bf16* v_s = sh.kv[wave][1];
  const int ug = blockIdx.y, b = ug / P.units, u = ug % P.units;
  const int hk = (P.units == P.hk) ? u : u / P.g;
  const int head0 = (P.units == P.hk) ? u * P.g : u;
  const int wid = bx * kDecodeWaves + wave, nw = P.nsplit * kDecodeWaves;

  bf16x8 Qf[KS];
  {
    const bool okq = n_ < P.gc;
    const __bf16* qp = q + b * P.sq[0] + (long)(head0 + (okq ? n_ : 0)) * P.sq[1] + 8 * h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) Qf[ks] = okq ? load8(qp + 16 * ks) : zero_frag();
  }
  const float sc = P.scale * kLog2e;

  float (&step_s)[2][64] = sh.step;
  int* sel_s = sh.sel;
  bool fresh = false;                  // kNewToken: this launch brings a token that the caches have room for
  int new_row = -1;
  if constexpr (ROLE == kNewToken) {
    const int pos = P.dyn != nullptr ? P.dyn[0] : P.start + P.count - 1;
    fresh = pos >= 0 && (P.dyn == nullptr || pos < P.cap_len);
    if (threadIdx.x < D / 2) {
      const float f = A.nt.freqs_bf16 ? (float)reinterpret_cast<const __bf16*>(A.nt.freqs)[threadIdx.x] : reinterpret_cast<const float*>(A.nt.freqs)[threadIdx.x];
      sincosf((float)pos * f, &step_s[1][threadIdx.x], &step_s[0][threadIdx.x]);
    }
    __syncthreads();
    auto rotate = [&](bf16x8 x, int pair0) {
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float cs = step_s[0][pair0 + e], sn = step_s[1][pair0 + e], a = (float)x[2 * e], c = (float)x[2 * e + 1];
        o[2 * e] = (__bf16)(a * cs - c * sn);
        o[2 * e + 1] = (__bf16)(c * cs + a * sn);
      }
      return o;
    };
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) Qf[ks] = rotate(Qf[ks], 8 * ks + 4 * h);
    if (wid == 0 && n_ < P.gc) {
      __bf16* rq = A.nt.rq + ((long)b * P.hk * P.g + head0 + n_) * D + 8 * h;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) *reinterpret_cast<bf16x8*>(rq + 16 * ks) = Qf[ks];
    }
    new_row = (P.count - 1) & 31;      // of the last tile
  }
  if constexpr (ROLE == kTopk) {
    if (P.S > 0) {
      const int nb = P.dyn != nullptr ? min(max(P.dyn[1], 0), P.cap_nc) / A.topk.per_block : A.topk.nb;
      if (wave == 0)
        wave_topk(A.topk.pooled + (long)ug * A.topk.stride, nb, P.S, lane, step_s[0], reinterpret_cast<int*>(step_s[1]), sel_s,
                  bx == 0 ? A.topk.idx + (long)ug * A.topk.kstride : nullptr, A.topk.fm + (long)ug * A.topk.kstride);
      __syncthreads();
    }
  }

  float m = -INFINITY, l = 0.f;
  floatx16 Oa[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) Oa[dt] = zero_acc();

  // rows are fetched with whole-row coalesced loads (LPR lanes per row) one tile ahead of the
  // arithmetic, and turned into MFMA operands through the wave's private LDS tiles
  bf16x8 kr[NI], vr[NI];
  auto issue = [&](const DecodeTile& T) {
#pragma unroll
    for (int r = 0; r < NI; ++r) {
      const int row = RPI * r + lr;
      const long rc = row < T.nvalid ? row : 0;
      kr[r] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(T.kb + rc * T.ks + 8 * lc));      // every cached row is read once per step
      vr[r] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(T.vb + rc * T.vs + 8 * lc));
    }
  };
  auto next_tile = [&](int t, DecodeTile& T) {
    for (; t < P.tiles; t += nw) {
      T = decode_tile(P, D, t, b, hk, ug, k, v, mem_k, mem_v, idx, fmask, ROLE == kTopk ? sel_s : nullptr);
      if (T.nvalid > 0) break;
    }
    return t;
  };

  DecodeTile T, Tn;
  int t = next_tile(wid, T);
  if (t < P.tiles) issue(T);
  while (t < P.tiles) {
    if constexpr (ROLE == kNewToken) {
      if (fresh && t == P.tiles - 1) {
        // the newest key and value: from the projection into this tile (the rows just read are not written yet), the caches
        // and the open compression window
        // (rows past it repeat it: they were read in its place)
        const NewToken& N = A.nt;
        const bf16x8 kx = load8(N.k + b * N.k0 + hk * N.k1 + 8 * lc), vx = load8(N.v + b * N.v0 + hk * N.v1 + 8 * lc);
        bf16x8 ko;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float cs = step_s[0][4 * lc + e], sn = step_s[1][4 * lc + e], a = (float)kx[2 * e], c = (float)kx[2 * e + 1];
          ko[2 * e] = (__bf16)(a * cs - c * sn);
          ko[2 * e + 1] = (__bf16)(c * cs + a * sn);
        }
#pragma unroll
        for (int r = 0; r < NI; ++r)
          if (RPI * r + lr >= new_row) { kr[r] = ko; vr[r] = vx; }
        if (lr == new_row % RPI) {
          const long row = P.start + P.count - 1;
          *reinterpret_cast<bf16x8*>(N.kc + b * P.sk[0] + hk * P.sk[1] + row * P.sk[2] + 8 * lc) = ko;
          *reinterpret_cast<bf16x8*>(N.vc + b * P.sv[0] + hk * P.sv[1] + row * P.sv[2] + 8 * lc) = vx;
          if (N.krun != nullptr) {
            const long at = N.ring > 0 ? row % N.ring : 0;
            *reinterpret_cast<bf16x8*>(N.krun + b * N.ku0 + hk * N.ku1 + at * N.ku_row + 8 * lc) = kx;
            *reinterpret_cast<bf16x8*>(N.vrun + b * N.vu0 + hk * N.vu1 + at * N.vu_row + 8 * lc) = vx;
          }
        }
      }
    }
#pragma unroll
    for (int r = 0; r < NI; ++r) {
      *reinterpret_cast<bf16x8*>(k_s + (RPI * r + lr) * RS + 8 * lc) = kr[r];
      *reinterpret_cast<bf16x8*>(v_s + (RPI * r + lr) * RSV + 8 * lc) = vr[r];
    }
    const int tn = next_tile(t + nw, Tn);
    if (tn < P.tiles) issue(Tn);
    __builtin_amdgcn_sched_barrier(0);

    floatx16 Sa = zero_acc();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) Sa = mfma32(lds_row_operand(k_s, RS, ks, lane), Qf[ks], Sa);
    if constexpr (ROLE == kPooled)
      if (T.lcol >= 0) pool_tile(P, A.pool, Sa, T.lcol, A.pool.share ? (long)ug : (long)b * P.hk * P.g + head0 + n_, n_, h);

    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int kl = 8 * (i >> 2) + 4 * h + (i & 3);
      if (ROLE == kPlain && logits != nullptr && T.lcol >= 0 && n_ < P.gc && kl < T.nvalid)
        logits[((long)b * P.hk * P.g + head0 + n_) * P.lstride + T.lcol + kl] = Sa[i] * P.scale;
      const float s = kl < T.nvalid ? Sa[i] * sc : -INFINITY;
      Sa[i] = s;
      mx = fmaxf(mx, s);
    }
    mx = halves_max(mx);
    const float mn = fmaxf(m, mx);
    const float alpha = fast_exp2(m - mn);
    float ls = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = fast_exp2(Sa[i] - mn);
      Sa[i] = p;
      ls += p;
    }
    l = l * alpha + ls;
    m = mn;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) Oa[dt][i] *= alpha;
#pragma unroll
      for (int u2 = 0; u2 < 2; ++u2)
        Oa[dt] = mfma32(lds_transposed_operand(v_s, RSV, 16 * u2, 32 * dt, lane), pack8(Sa, 8 * u2), Oa[dt]);
    }
    t = tn;
    T = Tn;
  }
  l = halves_sum(l);

  // partial record of this wave: [gc][D] O, [gc] max, [gc] sum
  if (n_ < P.gc) {
    float* rec = part + ((long)ug * P.nparts + wid) * P.rec;
    if (h == 0) { rec[P.gc * D + n_] = m; rec[P.gc * D + P.gc + n_] = l; }
    float* o = rec + n_ * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        floatx4 w = {Oa[dt][4 * i4], Oa[dt][4 * i4 + 1], Oa[dt][4 * i4 + 2], Oa[dt][4 * i4 + 3]};
        *reinterpret_cast<floatx4*>(o + 32 * dt + 8 * i4 + 4 * h) = w;
      }
  }
}

template <int D, int ROLE>
__global__ __launch_bounds__(64 * kDecodeWaves) __attribute__((amdgpu_waves_per_eu(2))) void decode_attend_kernel(const AttendArgs A) {
  __shared__ DecodeShared<D> sh;
  decode_attend_body<D, ROLE>(A, blockIdx.x, sh);
}

// The compressed keys and the sliding window of a step, which do not depend on each other, in one launch: the work-groups of
// the second follow those of the first along x, so the short branch fills the chip while the long one drains.
template <int D, int ROLE>
__global__ __launch_bounds__(64 * kDecodeWaves) __attribute__((amdgpu_waves_per_eu(2))) void decode_attend_pair_kernel(const AttendArgs A, const AttendArgs B) {
  __shared__ DecodeShared<D> sh;
  if ((int)blockIdx.x < A.P.nsplit) decode_attend_body<D, ROLE>(A, blockIdx.x, sh);
  else decode_attend_body<D, kNewToken>(B, blockIdx.x - A.P.nsplit, sh);
}

// Log-sum-exp merge of the split-K partials of head (b, head) of one branch by a work-group of D threads: the
// partials' maxima and sums are read by one thread each and reduced through LDS, then thread f accumulates
// feature f over the partials that carry weight (loads independent of each other, so they overlap).
constexpr int kMaxParts = 64 * kDecodeWaves;

template <int D>
__device__ __forceinline__ float merge_head_partials(const DecodePlan& P, const float* __restrict__ part, int b, int head, int f,
                                                     float* w_s, float* red_s) {
  const int u = (P.units == P.hk) ? head / P.g : head, gi = (P.units == P.hk) ? head % P.g : 0;
  const float* base = part + (long)(b * P.units + u) * P.nparts * P.rec;
  const int om = P.gc * D + gi, ol = om + P.gc;
  constexpr int PT = (kMaxParts + D - 1) / D;          // partials per thread
  float mp[PT], lp[PT];
  float M = -INFINITY;
#pragma unroll
  for (int r = 0; r < PT; ++r) {
    const int p = f + r * D;
    mp[r] = p < P.nparts ? base[(long)p * P.rec + om] : -INFINITY;
    lp[r] = p < P.nparts ? base[(long)p * P.rec + ol] : 0.f;
    M = fmaxf(M, mp[r]);
  }
  auto block_reduce = [&](float v, bool is_max) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const float t = __shfl_xor(v, o, 64);
      v = is_max ? fmaxf(v, t) : v + t;
    }
    if (D > 64) {
      __syncthreads();
      if ((f & 63) == 0) red_s[f >> 6] = v;
      __syncthreads();
      v = red_s[0];
#pragma unroll
      for (int w = 1; w < D / 64; ++w) v = is_max ? fmaxf(v, red_s[w]) : v + red_s[w];
    }
    return v;
  };
  M = block_reduce(M, true);
  const bool any = M > -INFINITY;                      // false: no wave saw a key
  float L = 0.f;
  __syncthreads();                                     // w_s may still be read for the previous branch
#pragma unroll
  for (int r = 0; r < PT; ++r) {
    const int p = f + r * D;
    const float w = any ? fast_exp2(mp[r] - M) : 0.f;  // exp2(-inf) = 0 for waves that saw no key
    if (p < P.nparts) w_s[p] = w;
    L += w * lp[r];
  }
  L = block_reduce(L, false);
  __syncthreads();
  float acc = 0.f;
  // every wave wrote a finite record (zeros when it saw no key), so the loads need no guard and overlap
#pragma unroll 8
  for (int p = 0; p < P.nparts; ++p) acc += w_s[p] * base[(long)p * P.rec + gi * D + f];
  return L > 0.f ? acc / L : 0.f;
}

// one work-group per query head, one thread per feature
template <int D>
__global__ __launch_bounds__(D) void decode_merge_kernel(const DecodePlan P, const float* __restrict__ part, __bf16* __restrict__ out) {
  __shared__ float w_s[kMaxParts], red_s[4];
  const int hq = P.hk * P.g;
  const int bh = blockIdx.x, b = bh / hq, head = bh % hq;
  out[(long)bh * D + threadIdx.x] = (__bf16)merge_head_partials<D>(P, part, b, head, threadIdx.x, w_s, red_s);
}

// Merge of the three branches' partials, sigmoid strategy gate and head merge in one pass
// (NSA.py:534-545): out[b, head*D + f] = sum_s sigmoid(logit[b, 3*head + s]) * branch_s.
// A branch without a workspace (no compressed key cached yet) contributes zero.  `advance` (optional): the step's
// position counter, incremented here once every attention kernel of the step has run.
struct CombineArgs {
  DecodePlan P[3];
  const float* part[3];
  int* advance;
  long gate_row;                 // elements between the gate logits of consecutive batch rows
  const __bf16* gate_bias;       // optional [3 * heads], added to the logits (a projection computed without its bias)
};

// A work-group per query head, two waves per branch: every wave reduces the maxima and sums of its branch's partials itself
// (two per lane at most) and the branch's 2 x 64 lanes read the partials' features 16 bytes at a time, 256 / (D / 4) of them
// at once - three dependent rounds of memory whatever the number of partials.  (One thread per feature, one branch after
// the other with four barriers each: 10.9 us for 32 heads at 32k context.)
template <int D>
__global__ __launch_bounds__(384) void decode_combine_kernel(const CombineArgs A, const __bf16* __restrict__ gate_logits, __bf16* __restrict__ out) {
  constexpr int LPP = D / 4, PPR = 128 / LPP;              // lanes per partial, partials per round of a branch
  __shared__ float w_s[3][kMaxParts], sum_s[3];
  __shared__ __align__(16) float acc_s[3][PPR][D];
  const int hq = A.P[0].hk * A.P[0].g;
  const int bh = blockIdx.x, b = bh / hq, head = bh % hq;
  const int s = threadIdx.x >> 7, t = threadIdx.x & 127, lane = t & 63;
  const DecodePlan& P = A.P[s];
  if (A.part[s] != nullptr) {
    const int u = (P.units == P.hk) ? head / P.g : head, gi = (P.units == P.hk) ? head % P.g : 0;
    const float* base = A.part[s] + (long)(b * P.units + u) * P.nparts * P.rec;
    const int om = P.gc * D + gi, ol = om + P.gc;
    constexpr int PT = kMaxParts / 64;
    float mp[PT], lp[PT], M = -INFINITY, L = 0.f;
#pragma unroll
    for (int r = 0; r < PT; ++r) {
      const int p = lane + 64 * r;
      mp[r] = p < P.nparts ? base[(long)p * P.rec + om] : -INFINITY;
      lp[r] = p < P.nparts ? base[(long)p * P.rec + ol] : 0.f;
      M = fmaxf(M, mp[r]);
    }
    M = wave_reduce_max(M);
    const float ref = M > -INFINITY ? M : 0.f;             // no wave saw a key: every weight exp2(-inf) = 0
#pragma unroll
    for (int r = 0; r < PT; ++r) { mp[r] = fast_exp2(mp[r] - ref); L += mp[r] * lp[r]; }
    L = wave_reduce_sum(L);
    const float inv = L > 0.f ? 1.0f / L : 0.f;
    if (t < 64) {
      if (lane == 0) sum_s[s] = L;
#pragma unroll
      for (int r = 0; r < PT; ++r) w_s[s][lane + 64 * r] = mp[r] * inv;
    }
  }
  __syncthreads();
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  if (A.part[s] != nullptr) {
    const int u = (P.units == P.hk) ? head / P.g : head, gi = (P.units == P.hk) ? head % P.g : 0;
    const float* base = A.part[s] + (long)(b * P.units + u) * P.nparts * P.rec + gi * D + 4 * (t % LPP);
    // every wave of the attend kernels wrote its record (zeros when it saw no key), so the loads need no guard and overlap
#pragma unroll 8
    for (int p = t / LPP; p < P.nparts; p += PPR) acc += w_s[s][p] * *reinterpret_cast<const floatx4*>(base + (long)p * P.rec);
  }
  *reinterpret_cast<floatx4*>(&acc_s[s][t / LPP][4 * (t % LPP)]) = acc;
  __syncthreads();
  if (threadIdx.x < D) {
    const int f = threadIdx.x;
    float res = 0.f;
#pragma unroll
    for (int br = 0; br < 3; ++br) {
      if (A.part[br] == nullptr) continue;
      float o = 0.f;
#pragma unroll
      for (int r = 0; r < PPR; ++r) o += acc_s[br][r][f];
      o = sum_s[br] > 0.f ? o : 0.f;                       // no key, or a sum that is no number: nothing, as merge_head_partials
      float gl = (float)gate_logits[(long)b * A.gate_row + head * 3 + br];
      if (A.gate_bias != nullptr) gl += (float)A.gate_bias[head * 3 + br];
      res += (float)(__bf16)o / (1.f + __expf(-gl));       // branch outputs are rounded to bf16 as when each is merged on its own
    }
    out[(long)bh * D + f] = (__bf16)res;
  }
  if (A.advance != nullptr && blockIdx.x == 0 && threadIdx.x == 0) A.advance[0] += 1;
}

// `step`: the branch is one of a whole step's; `beside`: tiles of the other key range in its launch
static int make_decode_plan(const nsa_decode_desc* dsc, DecodePlan& P, bool step = false, int beside = 0) {
  if (!dsc) return NSA_E_ARG;
  P = DecodePlan{};
  P.b = dsc->batch; P.hk = dsc->kv_heads; P.g = dsc->group; P.d = dsc->dim_head;
  if (P.b <= 0 || P.hk <= 0 || P.g <= 0) return NSA_E_ARG;
  if (P.d != 64 && P.d != 128) return NSA_E_UNSUPPORTED;
  if (P.g > 32) return NSA_E_UNSUPPORTED;
  P.mode = dsc->mode;
  P.scale = dsc->scale;
  P.idx64 = dsc->idx_is_int64;
  for (int i = 0; i < 2; ++i) P.sq[i] = dsc->q_stride[i];
  for (int i = 0; i < 3; ++i) { P.sk[i] = dsc->k_stride[i]; P.sv[i] = dsc->v_stride[i]; }
  if ((P.sq[0] | P.sq[1] | P.sk[0] | P.sk[1] | P.sk[2] | P.sv[0] | P.sv[1] | P.sv[2]) & 7) return NSA_E_ARG;
  if (P.mode == 0) {
    P.start = dsc->start; P.count = dsc->count; P.mem = dsc->num_mem;
    if (P.start < 0 || P.count < 0 || P.mem < 0) return NSA_E_ARG;
    P.units = P.hk; P.gc = P.g;
    P.tiles = (P.mem + 31) / 32 + (P.count + 31) / 32;
  } else if (P.mode == 1) {
    P.B = dsc->block; P.S = dsc->num_sel; P.kv_len = dsc->kv_len;
    if (P.B < 1 || P.S < 0 || P.kv_len < 1) return NSA_E_ARG;
    const bool per_head = dsc->per_head_sel != 0;
    P.units = per_head ? P.hk * P.g : P.hk;
    P.gc = per_head ? 1 : P.g;
    P.tps = (P.B + 31) / 32;
    P.tiles = (P.S + 1) * P.tps;
  } else {
    return NSA_E_ARG;
  }
  const long units = (long)P.b * P.units;
  if (units > 65535) return NSA_E_UNSUPPORTED;
  // split-K: two tiles per wave, at most 4096 work-groups.  In a whole step - key ranges: two tiles per wave while that leaves
  // CUs without a work-group, else four (a partial record is written and read again for every wave), at most 2048
  // work-groups; selected blocks: a tile per wave (a chain of dependent loads: index, row) but at most 768 work-groups,
  // since each of them makes the selection for itself.  Measured at 32k context, microseconds a step, {2, 2} tiles and 4096
  // work-groups for both before: batch 1 41.7 -> 40.3 (4 tiles: 44.0), batch 8 60.0 -> 57.2, batch 32 141 -> 125.7; 16 heads
  // x 64, 8k context, batch 32: 44.4 -> 39.1.
  const int per4 = (P.tiles + 4 * kDecodeWaves - 1) / (4 * kDecodeWaves);
  const int tpw = !step ? 2 : P.mode == 1 ? 1 : (units * per4 >= 256 ? 4 : 2);
  const long most = !step ? 4096 : P.mode == 1 ? 768 : 2048;
  int ns = (P.tiles + tpw * kDecodeWaves - 1) / (tpw * kDecodeWaves);
  const long cap = units >= most ? 1 : most / units;
  if (ns > cap) ns = (int)cap;
  // The two key ranges of a step in wide heads: no more work-groups than the chip holds at once (four to a CU).  A second and
  // third round, begun where the first drains, cost more than the longer walks: 16 steps at 32k context, 32 heads x 128, batch 32
  // (2816 work-groups -> 1024) 2290 -> 2165 us, batch 16 (1792 -> 1024) 1640 -> 1555; 4000 tokens of context, batch 32 1580 -> 1542.
  // (At 64 features a work-group takes half as much, and the limit above is the better one.)
  if (step && P.mode == 0 && P.d == 128) {
    auto groups = [&](int tiles, int t) { return (tiles + t * kDecodeWaves - 1) / (t * kDecodeWaves); };
    for (int t = tpw; ns > 1 && (groups(P.tiles, t) + groups(beside, t)) * units > 1024; ++t) ns = groups(P.tiles, t + 1);
  }
  if (ns > 64) ns = 64;
  if (ns < 1) ns = 1;
  P.nsplit = ns; P.nparts = ns * kDecodeWaves;
  P.rec = P.gc * P.d + ((2 * P.gc + 3) & ~3);
  P.sstride = P.S; P.lstride = P.count;
  return 0;
}

static int check_attend(const DecodePlan& P, const void* q, const void* k, const void* v, const void* mem_k, const void* mem_v,
                        const void* idx, const uint8_t* fmask, void* ws, size_t ws_bytes) {
  if (!q || !ws) return NSA_E_ARG;
  if (P.mode == 0 && ((P.count > 0 && (!k || !v)) || (P.mem > 0 && (!mem_k || !mem_v)))) return NSA_E_ARG;
  if (P.mode == 1 && (!k || !v || (P.S > 0 && (!idx || !fmask)))) return NSA_E_ARG;
  if (ws_bytes < (size_t)P.b * P.units * P.nparts * P.rec * sizeof(float)) return NSA_E_WORKSPACE;
  return 0;
}

static AttendArgs attend_args(const DecodePlan& P, const void* q, const void* k, const void* v, const void* mem_k, const void* mem_v,
                              const void* idx, const uint8_t* fmask, void* ws, float* logits) {
  AttendArgs A{};
  A.P = P;
  A.q = (const __bf16*)q; A.k = (const __bf16*)k; A.v = (const __bf16*)v; A.mem_k = (const __bf16*)mem_k; A.mem_v = (const __bf16*)mem_v;
  A.idx = idx; A.fmask = fmask; A.part = (float*)ws; A.logits = logits;
  return A;
}

static int launch_attend(const DecodePlan& P, const void* q, const void* k, const void* v, const void* mem_k, const void* mem_v, const void* idx,
                         const uint8_t* fmask, void* ws, size_t ws_bytes, void* out, float* logits, void* stream) {
  if (int e = check_attend(P, q, k, v, mem_k, mem_v, idx, fmask, ws, ws_bytes)) return e;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid(P.nsplit, P.b * P.units);
  const int heads = P.b * P.hk * P.g;
  const AttendArgs A = attend_args(P, q, k, v, mem_k, mem_v, idx, fmask, ws, logits);
  if (P.d == 64) {
    hipLaunchKernelGGL((decode_attend_kernel<64, kPlain>), grid, dim3(64 * kDecodeWaves), 0, st, A);
    if (out) hipLaunchKernelGGL((decode_merge_kernel<64>), dim3(heads), dim3(64), 0, st, P, (const float*)ws, (__bf16*)out);
  } else {
    hipLaunchKernelGGL((decode_attend_kernel<128, kPlain>), grid, dim3(64 * kDecodeWaves), 0, st, A);
    if (out) hipLaunchKernelGGL((decode_merge_kernel<128>), dim3(heads), dim3(128), 0, st, P, (const float*)ws, (__bf16*)out);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

// One branch of a step in a role of its own; partials only (merged later by the combine kernel).
template <int ROLE>
static int launch_attend_role(const AttendArgs& A, size_t ws_bytes, void* stream) {
  if (int e = check_attend(A.P, A.q, A.k, A.v, A.mem_k, A.mem_v, A.idx, A.fmask, A.part, ws_bytes)) return e;
  const dim3 grid(A.P.nsplit, A.P.b * A.P.units);
  hipStream_t st = (hipStream_t)stream;
  if (A.P.d == 64) hipLaunchKernelGGL((decode_attend_kernel<64, ROLE>), grid, dim3(64 * kDecodeWaves), 0, st, A);
  else hipLaunchKernelGGL((decode_attend_kernel<128, ROLE>), grid, dim3(64 * kDecodeWaves), 0, st, A);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

// compressed keys (A, role kPooled or kPlain) and sliding window (B) over the same (batch, kv head) units in one launch
template <int ROLE>
static int launch_attend_pair(const AttendArgs& A, size_t wsa_bytes, const AttendArgs& B, size_t wsb_bytes, void* stream) {
  if (int e = check_attend(A.P, A.q, A.k, A.v, A.mem_k, A.mem_v, A.idx, A.fmask, A.part, wsa_bytes)) return e;
  if (int e = check_attend(B.P, B.q, B.k, B.v, B.mem_k, B.mem_v, B.idx, B.fmask, B.part, wsb_bytes)) return e;
  if (A.P.b * A.P.units != B.P.b * B.P.units || A.P.d != B.P.d) return NSA_E_ARG;
  const dim3 grid(A.P.nsplit + B.P.nsplit, A.P.b * A.P.units);
  hipStream_t st = (hipStream_t)stream;
  if (A.P.d == 64) hipLaunchKernelGGL((decode_attend_pair_kernel<64, ROLE>), grid, dim3(64 * kDecodeWaves), 0, st, A, B);
  else hipLaunchKernelGGL((decode_attend_pair_kernel<128, ROLE>), grid, dim3(64 * kDecodeWaves), 0, st, A, B);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

static int launch_combine(const DecodePlan* plans[3], const void* const ws[3], const void* gate_logits, int64_t gate_row, const void* gate_bias,
                          void* out, int* advance, void* stream) {
  if (!gate_logits || !out) return NSA_E_ARG;
  CombineArgs A;
  A.advance = advance;
  int ref = -1;
  for (int s = 0; s < 3; ++s) {
    A.part[s] = nullptr;
    A.P[s] = DecodePlan{};
    if (!ws[s]) continue;
    A.P[s] = *plans[s];
    A.part[s] = (const float*)ws[s];
    if (ref < 0) ref = s;
    else if (A.P[s].b != A.P[ref].b || A.P[s].hk != A.P[ref].hk || A.P[s].g != A.P[ref].g || A.P[s].d != A.P[ref].d) return NSA_E_ARG;
  }
  if (ref < 0) return NSA_E_ARG;
  if (ref != 0) A.P[0] = A.P[ref];         // the kernel reads the head counts from slot 0
  A.gate_row = gate_row > 0 ? (long)gate_row : 3L * A.P[ref].hk * A.P[ref].g;
  A.gate_bias = (const __bf16*)gate_bias;
  const int heads = A.P[ref].b * A.P[ref].hk * A.P[ref].g;
  hipStream_t st = (hipStream_t)stream;
  if (A.P[ref].d == 64)
    hipLaunchKernelGGL((decode_combine_kernel<64>), dim3(heads), dim3(384), 0, st, A, (const __bf16*)gate_logits, (__bf16*)out);
  else
    hipLaunchKernelGGL((decode_combine_kernel<128>), dim3(heads), dim3(384), 0, st, A, (const __bf16*)gate_logits, (__bf16*)out);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}


}  // namespace nsa

namespace nsa {
static int decode_partials_bytes(const nsa_decode_desc* dsc, size_t* bytes, bool step, int beside = 0) {
  DecodePlan P;
  if (int e = make_decode_plan(dsc, P, step, beside)) return e;
  if (!bytes) return NSA_E_ARG;
  *bytes = (size_t)P.b * P.units * P.nparts * P.rec * sizeof(float);
  return 0;
}
}  // namespace nsa

extern "C" int nsa_decode_workspace_bytes(const nsa_decode_desc* dsc, size_t* bytes) { return nsa::decode_partials_bytes(dsc, bytes, false); }

extern "C" int nsa_decode_attend(const nsa_decode_desc* dsc, const void* q, const void* k, const void* v, const void* mem_k,
                                 const void* mem_v, const void* idx, const uint8_t* fmask, void* ws, size_t ws_bytes, void* out,
                                 float* logits, void* stream) {
  using namespace nsa;
  DecodePlan P;
  if (int e = make_decode_plan(dsc, P)) return e;
  return launch_attend(P, q, k, v, mem_k, mem_v, idx, fmask, ws, ws_bytes, out, logits, stream);
}

// ------------------------------------------------------------------------------------------------------------
// nsa_decode_attend for callers that cannot allocate (a stream under graph capture, a serving loop that forbids
// hipMalloc): the split-K partials go to a fixed device array of this library instead of a caller workspace.
// Every GPU the library runs on holds its own copy of the array, at its own address, until the process ends; in
// host code the array's name is only a handle, so the address is looked up once per device with
// hipGetSymbolAddress and that pointer is what the kernels receive.  All calls on a GPU share the array: calls
// that overlap on one GPU (two streams, two threads) race.  Nothing has to be cleared between calls: every wave
// of the attend kernel writes its partial record (a neutral one when it has no tile) before the merge reads it.
#include <mutex>

namespace nsa {
constexpr size_t kNoAllocScratchBytes = NSA_DECODE_NOALLOC_SCRATCH_BYTES;
constexpr int kNoAllocMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
static void* g_scratch_ptr[kNoAllocMaxDevices];       // per device: device address of `scratch`
static std::mutex g_scratch_mutex;

static int scratch_of_current_device(void** ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kNoAllocMaxDevices) return NSA_E_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return NSA_E_ARG;
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return 0;
}
}  // namespace nsa

extern "C" int nsa_decode_attend_noalloc(const nsa_decode_desc* dsc, const void* q, const void* k, const void* v, const void* mem_k,
                                         const void* mem_v, const void* idx, const uint8_t* fmask, void* out, float* logits, void* stream) {
  using namespace nsa;
  DecodePlan P;
  if (int e = make_decode_plan(dsc, P)) return e;
  if (!out) return NSA_E_ARG;                          // the partials are private to the library: the merged output is the result
  const size_t need = (size_t)P.b * P.units * P.nparts * P.rec * sizeof(float);
  if (need > kNoAllocScratchBytes) return NSA_E_WORKSPACE;
  void* ws = nullptr;
  if (int e = scratch_of_current_device(&ws)) return e;
  return launch_attend(P, q, k, v, mem_k, mem_v, idx, fmask, ws, kNoAllocScratchBytes, out, logits, stream);
}

extern "C" int nsa_decode_combine(const nsa_decode_desc* compressed, const void* ws_compressed, const nsa_decode_desc* selected,
                                  const void* ws_selected, const nsa_decode_desc* sliding, const void* ws_sliding,
                                  const void* gate_logits, void* out, void* stream) {
  using namespace nsa;
  const nsa_decode_desc* dsc[3] = {compressed, selected, sliding};
  const void* ws[3] = {ws_compressed, ws_selected, ws_sliding};
  DecodePlan P[3];
  const DecodePlan* pp[3] = {&P[0], &P[1], &P[2]};
  for (int s = 0; s < 3; ++s)
    if (ws[s])
      if (int e = make_decode_plan(dsc[s], P[s])) return e;
  return launch_combine(pp, ws, gate_logits, 0, nullptr, out, nullptr, stream);
}

// ---------------------------------------------------------------------------- whole step
// The attention part of one decode step as a single host call and three launches: the sliding branch, which rotates the queries
// and brings the new token into the caches, together with the compressed branch, which leaves its logits pooled per block; the
// selected-block branch, whose work-groups make the selection themselves; merge + gate.  (Blocks of other than 1, 2, 4 .. 32
// compressed keys: one logit per key and head, and the top-k kernel as a launch of its own.)

namespace nsa {

struct StepLayout {
  nsa_decode_desc c, f, s;
  int nb, k;                       // selection blocks available / selected this step
  int sel_units;                   // rows of idx per batch element
  int tiles_c, tiles_s;            // 32-key tiles of the two key ranges
  int pooled;                      // the compressed branch leaves pooled logits and the selected-block branch selects
  size_t off_rq, off_wsc, off_wsf, off_wss, off_logits, off_idx, off_vals, off_fm, total;
  size_t wsc, wsf, wss;
};

static size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }

static int make_step_layout(const nsa_decode_step_desc* d, StepLayout& L) {
  if (!d) return NSA_E_ARG;
  if (d->batch <= 0 || d->heads <= 0 || d->kv_heads <= 0 || d->heads % d->kv_heads) return NSA_E_ARG;
  if (d->pos < 0 || d->num_compressed < 0 || d->num_mem < 0 || d->per_block <= 0 || d->block <= 0 || d->num_sel < 0 || d->window < 0)
    return NSA_E_ARG;
  const int g = d->heads / d->kv_heads, kv_len = d->pos + 1;
  auto common = [&](nsa_decode_desc& x) {
    x = nsa_decode_desc{};
    x.batch = d->batch; x.kv_heads = d->kv_heads; x.group = g; x.dim_head = d->dim_head; x.scale = d->scale;
  };
  // compressed branch reads the un-rotated projection, the other two the rotated queries in the workspace
  common(L.c);
  L.c.mode = 0; L.c.start = 0; L.c.count = d->num_compressed; L.c.num_mem = d->num_compressed > 0 ? d->num_mem : 0;
  L.c.q_stride[0] = d->q_stride[0]; L.c.q_stride[1] = d->q_stride[1];
  for (int i = 0; i < 3; ++i) { L.c.k_stride[i] = d->ck_stride[i]; L.c.v_stride[i] = d->cv_stride[i]; }
  L.nb = d->num_compressed / d->per_block;
  L.k = d->num_sel < L.nb ? d->num_sel : L.nb;
  L.sel_units = d->share ? d->kv_heads : d->heads;
  common(L.f);
  L.f.mode = 1; L.f.block = d->block; L.f.num_sel = L.k; L.f.kv_len = kv_len; L.f.per_head_sel = (!d->share && g > 1) ? 1 : 0;
  L.f.idx_is_int64 = 0;
  common(L.s);
  L.s.mode = 0;
  const int w = kv_len < d->window + 1 ? kv_len : d->window + 1;
  L.s.start = kv_len - w; L.s.count = w; L.s.num_mem = 0;
  for (nsa_decode_desc* x : {&L.f, &L.s}) {
    x->q_stride[0] = (int64_t)d->heads * d->dim_head; x->q_stride[1] = d->dim_head;
    for (int i = 0; i < 3; ++i) { x->k_stride[i] = d->kc_stride[i]; x->v_stride[i] = d->vc_stride[i]; }
  }
  auto tiles = [](const nsa_decode_desc& x) { return (x.num_mem + 31) / 32 + (x.count + 31) / 32; };
  L.tiles_c = d->num_compressed > 0 ? tiles(L.c) : 0;
  L.tiles_s = tiles(L.s);
  if (d->num_compressed > 0)
    if (int e = decode_partials_bytes(&L.c, &L.wsc, true, L.tiles_s)) return e;
  if (d->num_compressed <= 0) L.wsc = 0;
  if (int e = decode_partials_bytes(&L.f, &L.wsf, true)) return e;
  if (int e = decode_partials_bytes(&L.s, &L.wss, true, L.tiles_c)) return e;
  size_t o = 0;
  L.off_rq = o;     o = up256(o + (size_t)d->batch * d->heads * d->dim_head * 2);
  L.off_wsc = o;    o = up256(o + L.wsc);
  L.off_wsf = o;    o = up256(o + L.wsf);
  L.off_wss = o;    o = up256(o + L.wss);
  // one logit per block and selection row where a block is 1, 2, 4 .. 32 compressed keys (a 32-key tile pools them in
  // registers), else one per key and head, pooled by the top-k kernel
  L.pooled = d->per_block <= 32 && !(d->per_block & (d->per_block - 1));
  const size_t row = L.pooled ? (size_t)L.sel_units * (L.nb > 0 ? L.nb : 1) : (size_t)d->heads * (d->num_compressed > 0 ? d->num_compressed : 1);
  L.off_logits = o; o = up256(o + (size_t)d->batch * row * 4);
  const size_t sel = (size_t)d->batch * L.sel_units * (L.k > 0 ? L.k : 1);
  L.off_idx = o;    o = up256(o + sel * 4);
  L.off_vals = o;   o = up256(o + sel * 4);
  L.off_fm = o;     o = up256(o + sel);
  L.total = o;
  return 0;
}

}  // namespace nsa

extern "C" int nsa_decode_step_workspace_bytes(const nsa_decode_step_desc* desc, size_t* bytes, size_t* idx_offset, size_t* fmask_offset,
                                               int32_t* num_selected) {
  nsa::StepLayout L;
  if (int e = nsa::make_step_layout(desc, L)) return e;
  if (!bytes) return NSA_E_ARG;
  *bytes = L.total;
  if (idx_offset) *idx_offset = L.off_idx;
  if (fmask_offset) *fmask_offset = L.off_fm;
  if (num_selected) *num_selected = L.k;
  return 0;
}

// Declared in nsa_topk.hip: the top-k launch with lengths read from device memory.
namespace nsa {
int decode_topk_launch(const float* logits, int32_t batch, int32_t kv_heads, int32_t group, int32_t num_compressed, int32_t per_block,
                       int32_t share, int32_t k, int32_t* idx, float* vals, uint8_t* fmask, const int32_t* state, void* stream);

// The launches of a step.  state == nullptr: the lengths are the descriptor's; otherwise they are read from it when the
// kernels run and the descriptor's are capacities.  krun / vrun: the row for the new token (ring == 0) or a ring of rows.
int run_decode_step(const nsa_decode_step_desc* d, int32_t* state, const void* q, const void* k, const void* v, const void* freqs, int freqs_bf16,
                    void* k_cache, void* v_cache, const void* ck_cache, const void* cv_cache, const void* mem_k, const void* mem_v, void* krun, void* vrun,
                    int64_t krun_row, int64_t vrun_row, int32_t ring, const void* gate_logits, int64_t gate_row, const void* gate_bias, void* ws,
                    size_t ws_bytes, void* out, bool advance, void* stream) {
  StepLayout L;
  if (int e = make_step_layout(d, L)) return e;
  if (!q || !k || !v || !freqs || !k_cache || !v_cache || !gate_logits || !ws || !out) return NSA_E_ARG;
  if (ws_bytes < L.total) return NSA_E_WORKSPACE;
  const bool has_c = d->num_compressed > 0;
  if (has_c && (!ck_cache || !cv_cache)) return NSA_E_ARG;
  if ((d->k_stride[0] | d->k_stride[1] | d->v_stride[0] | d->v_stride[1]) & 7) return NSA_E_ARG;
  if (krun || vrun) {
    if (!krun || !vrun || ((d->krun_stride[0] | d->krun_stride[1] | d->vrun_stride[0] | d->vrun_stride[1]) & 7)) return NSA_E_ARG;
    if (ring > 0 && ((krun_row | vrun_row) & 7)) return NSA_E_ARG;
  }
  if (L.k > 0 && (L.nb > 64 * 32 || L.k > 64)) return NSA_E_UNSUPPORTED;
  DecodePlan Pc{}, Pf, Ps;
  if (has_c)
    if (int e = make_decode_plan(&L.c, Pc, true, L.tiles_s)) return e;
  if (int e = make_decode_plan(&L.f, Pf, true)) return e;
  if (int e = make_decode_plan(&L.s, Ps, true, L.tiles_c)) return e;
  if (state != nullptr) {
    int kind = 1;
    for (DecodePlan* P : {&Pc, &Pf, &Ps}) {
      P->dyn = state; P->dyn_kind = kind++;
      P->window = d->window; P->per_block = d->per_block; P->smax = L.k;
      P->cap_len = d->pos + 1; P->cap_nc = d->num_compressed;
    }
    Pc.lstride = d->num_compressed;
    Pf.sstride = L.k;
  }
  char* w = (char*)ws;
  void* rq = w + L.off_rq;
  float* logits = (float*)(w + L.off_logits);
  int32_t* idx = (int32_t*)(w + L.off_idx);
  uint8_t* fm = (uint8_t*)(w + L.off_fm);

  AttendArgs S = attend_args(Ps, q, k_cache, v_cache, nullptr, nullptr, nullptr, nullptr, w + L.off_wss, nullptr);
  for (int i = 0; i < 2; ++i) S.P.sq[i] = d->q_stride[i];                  // the projection's queries, rotated on the way in
  if ((S.P.sq[0] | S.P.sq[1]) & 7) return NSA_E_ARG;
  S.nt = NewToken{(const __bf16*)k, (const __bf16*)v, (long)d->k_stride[0], (long)d->k_stride[1], (long)d->v_stride[0], (long)d->v_stride[1], freqs, freqs_bf16,
                  (__bf16*)rq, (__bf16*)k_cache, (__bf16*)v_cache, (__bf16*)krun, (__bf16*)vrun, (long)d->krun_stride[0], (long)d->krun_stride[1],
                  (long)d->vrun_stride[0], (long)d->vrun_stride[1], (long)krun_row, (long)vrun_row, ring};
  if (has_c) {
    AttendArgs C = attend_args(Pc, q, ck_cache, cv_cache, mem_k, mem_v, nullptr, nullptr, w + L.off_wsc, L.pooled ? nullptr : logits);
    C.pool = PoolOut{logits, (long)(L.nb > 0 ? L.nb : 1), d->per_block, d->share ? 1 : 0};
    if (int e = L.pooled ? launch_attend_pair<kPooled>(C, L.wsc, S, L.wss, stream) : launch_attend_pair<kPlain>(C, L.wsc, S, L.wss, stream)) return e;
  } else if (int e = launch_attend_role<kNewToken>(S, L.wss, stream)) {
    return e;
  }
  AttendArgs F = attend_args(Pf, rq, k_cache, v_cache, nullptr, nullptr, L.k > 0 ? idx : nullptr, L.k > 0 ? fm : nullptr, w + L.off_wsf, nullptr);
  if (L.pooled) {
    F.topk = TopkIn{logits, (long)(L.nb > 0 ? L.nb : 1), L.nb, d->per_block, L.k, idx, fm};
    if (int e = launch_attend_role<kTopk>(F, L.wsf, stream)) return e;
  } else {
    if (L.k > 0)
      if (int e = decode_topk_launch(logits, d->batch, d->kv_heads, d->heads / d->kv_heads, d->num_compressed, d->per_block, d->share, L.k, idx,
                                     (float*)(w + L.off_vals), fm, state, stream))
        return e;
    if (int e = launch_attend_role<kPlain>(F, L.wsf, stream)) return e;
  }
  const DecodePlan* pp[3] = {&Pc, &Pf, &Ps};
  const void* wsp[3] = {has_c ? w + L.off_wsc : nullptr, w + L.off_wsf, w + L.off_wss};
  return launch_combine(pp, wsp, gate_logits, gate_row, gate_bias, out, advance ? state : nullptr, stream);
}
}  // namespace nsa

extern "C" int nsa_decode_step(const nsa_decode_step_desc* d, const void* q, const void* k, const void* v, const float* freqs,
                               void* k_cache, void* v_cache, const void* ck_cache, const void* cv_cache, const void* mem_k,
                               const void* mem_v, void* k_run_row, void* v_run_row, const void* gate_logits, void* ws, size_t ws_bytes,
                               void* out, void* stream) {
  return nsa::run_decode_step(d, nullptr, q, k, v, freqs, 0, k_cache, v_cache, ck_cache, cv_cache, mem_k, mem_v, k_run_row, v_run_row, 0, 0, 0, gate_logits, 0,
                       nullptr, ws, ws_bytes, out, false, stream);
}

extern "C" int nsa_decode_step_dyn(const nsa_decode_step_desc* cap, int32_t* state, const void* q, const void* k, const void* v,
                                   const float* freqs, void* k_cache, void* v_cache, const void* ck_cache, const void* cv_cache,
                                   const void* mem_k, const void* mem_v, void* k_run, void* v_run, int64_t krun_row_stride,
                                   int64_t vrun_row_stride, int32_t run_ring, const void* gate_logits, int64_t gate_row_stride,
                                   const void* gate_bias, void* ws, size_t ws_bytes, void* out, int32_t advance, void* stream) {
  if (!state || ((k_run || v_run) && run_ring <= 0)) return NSA_E_ARG;
  return nsa::run_decode_step(cap, state, q, k, v, freqs, 0, k_cache, v_cache, ck_cache, cv_cache, mem_k, mem_v, k_run, v_run, krun_row_stride, vrun_row_stride,
                       run_ring, gate_logits, gate_row_stride, gate_bias, ws, ws_bytes, out, advance != 0, stream);
}
