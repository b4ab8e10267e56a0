// fp32 forward kernels: the attention branches evaluated entirely in fp32 (products, softmax,
// accumulation), for fp32 modules, whose outputs must agree with the reference's fp32 torch path
// to its own test tolerance (1e-5, tests/test_sparse_attn.py:86).  The bf16 MFMA kernels cannot give
// that.  They follow the same contracts as nsa_select_fwd (NSA.py:741-819) and nsa_dense_fwd
// (NSA.py:153-184, 632-639, 841-850): any head dimension <= 128 that is a multiple of 4, any group
// size, any block size.
//
// Two kernels:
//  * f32_tile_kernel  - interval masks (band, strided prefix) and selections of a fair share of the blocks: 32 rows (query, head)
//    per wave against 32-key tiles shared by the work-group, on the bf16 matrix instructions with operands split in three;
//  * f32_rows_kernel  - one query of one kv head per wave (or per work-group) against 64-key tiles gathered
//    from anywhere, v_mfma_f32_4x4x1 with 16 blocks = 64 keys x 4 heads: block selection, and interval
//    masks with few queries (decode steps).
#include <type_traits>
#include <algorithm>
#include "nsa_split.hpp"
#include "../../include/nsa_hip.h"

namespace nsa {

constexpr int kF32MaxD = 128;

struct F32Args {
  int b, hk, bh, g, n, nk, d;          // n: number of queries (rows of q / out); nk: key rows after the memory slots
  int qoff;                       // query row i sits at sequence position i + qoff
  float scale;
  long sq[3], sk[3], sv[3];
  // dense
  int mode, causal, wb, wf, st, mem;
  const float *memk, *memv;       // the memory rows [hk, mem, d] when they are not the first rows of k / v, else null
  // selection
  int S, B, W, idx64, uniform, lb;      // lb: log2 of the block, where it is a power of two
};

// First and last key row (memory slots included, they are always visible) that the query at `pos` sees
__device__ __forceinline__ void f32_interval(const F32Args& A, int pos, int& lo, int& hi) {
  if (A.mode == 0) { lo = max(0, pos - A.wb); hi = min(A.nk - 1, pos + A.wf); }
  else { lo = 0; hi = A.mem + (A.causal ? min(A.nk - 1, pos / A.st - 1) : A.nk - 1); }
}

// ------------------------------------------------------------------------------------------ rows
//
// One query of one kv head, four of its heads at a time, against tiles of 64 gathered keys.
//   S = K Q^T: A = K (lane = key), B = Q (lane % 4 = head, the same in all 16 blocks) -> lane l holds head l % 4 of keys
//   4 (l / 4) + i in register i.  That is the A layout of the second product when block l / 4 is broadcast to all
//   blocks (cbsz = 4, abid = l / 4), so O += P V takes P's registers as they are: B = V (lane = feature), and the result
//   has lane = feature, register = head.
// K and V pass through LDS 64 rows x 64 features at a time (a lane needs whole key rows, the memory gives 16 bytes of four
// rows per instruction); the next piece is in flight while one is multiplied.  K pieces are stored with chunk c of row r at
// position c ^ (r % 16) (16-byte reads of 64 rows without bank conflicts), V pieces as they are.
// Bound by the vector memory path of the CU: a query and head group reads each of its K / V rows for itself, 32 KB per 64
// keys at d = 64, and they arrive at 27 bytes per cycle and CU (16.6 TB/s) whether they come from HBM, an L2 or - every
// query given the same block - the CU's own cache.  17 blocks of 64 keys, 4 heads, d = 64, 16384 queries: 0.52 ms
// (4.64 ms with lane = key dot products in scalar FMAs); one query at a time: 24 us (106 us).

constexpr int kRowsPiece = 64 * 64;      // floats of one wave's piece

template <int DT>
struct RowsState {
  float m, l;              // of head lane % 4; l: this lane's keys only
  floatx4 acc[DT];         // lane = feature, register = head
};

// max over the lanes of equal lane % 4
__device__ __forceinline__ float max_mod4(float v) {
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x124, 0xF, 0xF, true)));   // row_ror:4
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xF, 0xF, true)));   // row_ror:8
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return halves_max(v);
}
__device__ __forceinline__ float sum_mod4(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x124, 0xF, 0xF, true));
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xF, 0xF, true));
  v += __shfl_xor(v, 16, 64);
  return halves_sum(v);
}

struct RowsStage { floatx4 x[16]; };

// this lane's 16 bytes of rows 4 r + lane / 16, r = 0 .. 15, of the tile whose rows `rows_s` lists.  `special` (wave-uniform): some
// of them are padding keys (row -1: zeros) or memory rows of an array of their own (row -2 - m: row m of `mem`), or this piece's
// chunks reach past the head dimension (zeros).
template <bool FULL>
__device__ __forceinline__ void rows_load(RowsStage& st, const float* __restrict__ base, long stride, const float* __restrict__ mem, int d,
                                          const int* __restrict__ rows_s, int r0, int col, bool inside, bool special, int quarters) {
  const float* bc = base + (inside ? col : 0);
  if (!special) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (FULL || r < 4 || r / 4 < quarters) st.x[r] = *reinterpret_cast<const floatx4*>(bc + (long)rows_s[4 * r + r0] * stride);
  } else {
    const float* mc = mem + (inside ? col : 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = rows_s[4 * r + r0];
      const bool real = inside && row != -1;
      const float* p = row <= -2 ? mc + (long)(-2 - row) * d : bc + (long)max(row, 0) * stride;
      const floatx4 x = *reinterpret_cast<const floatx4*>(p);
#pragma unroll
      for (int e = 0; e < 4; ++e) st.x[r][e] = real ? x[e] : 0.f;
    }
  }
}

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// `total` keys; key(v) -> row of k / v (v < total), -1 for a padding key past the sequence end (logit 0, value 0), -2 - m for
// row m of mk / mv.  Tiles first, first + step, ...  `flat`: every key scores 0, whatever it holds.
template <int DT, class Key>
__device__ __forceinline__ void rows_walk(const F32Args& A, float* __restrict__ piece, int* __restrict__ rows_s, const float (&q)[DT][64], const float* __restrict__ kb,
                                          const float* __restrict__ vb, const float* __restrict__ mk, const float* __restrict__ mv, int total,
                                          int first, int step, bool flat, Key key, RowsState<DT>& S, int lane) {
  const int tiles = (total + 63) >> 6;
  if (first >= tiles) return;
  const int chunk = lane & 15, r0 = lane >> 4;
  bool special = false;
  // rows of tile t's keys; places behind the last key repeat it (their scores are masked)
  auto locate = [&](int t) {
    const int row = key(min(t * 64 + lane, total - 1));
    special = __any(row < 0);
    __builtin_amdgcn_wave_barrier();
    rows_s[lane] = row;
    __builtin_amdgcn_wave_barrier();
  };
  // A tile's rows move 16 at a time and the last tile leaves out those that no key needs (with small blocks it holds little but
  // the own block: 1 to 16 of 64 keys at a block of 16).  Rows of LDS that were left out hold old values: as keys they give scores
  // that are masked, as values they are not multiplied.  4 blocks of 16 keys and the own one, 2 heads, d = 64, 32768
  // queries: 195 -> 168 us; 17 blocks of 64 keys: the same as before (478 us, 16424 queries).
  // (The full tiles' code holds no branch for it: with one around every quarter 17 blocks of 64 keys took 4 % longer.)
  auto quarters_of = [&](int t) { return DT > 1 || special ? 4 : __builtin_amdgcn_readfirstlane((min(total - 64 * t, 64) + 15) >> 4); };
  int quarters = 4;
  RowsStage st;
  auto load_k = [&](auto full, int ft) {
    rows_load<decltype(full)::value>(st, kb, A.sk[2], mk, A.d, rows_s, r0, 64 * ft + 4 * chunk, 64 * ft + 4 * chunk < A.d, special || 64 * (ft + 1) > A.d, quarters);
  };
  auto load_v = [&](auto full, int ft) {
    rows_load<decltype(full)::value>(st, vb, A.sv[2], mv, A.d, rows_s, r0, 64 * ft + 4 * chunk, 64 * ft + 4 * chunk < A.d, special || 64 * (ft + 1) > A.d, quarters);
  };
  using Full = std::integral_constant<bool, true>;
  using Part = std::integral_constant<bool, false>;
  locate(first);
  quarters = quarters_of(first);
  if (DT > 1 || quarters == 4) load_k(Full{}, 0);
  else load_k(Part{}, 0);
  auto tile = [&](auto full, int t) {
    constexpr bool FULL = decltype(full)::value;
    const int here = quarters;                           // of tile t; `quarters` moves on with the loads
    floatx4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ft = 0; ft < DT; ++ft) {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (FULL || r < 4 || r / 4 < here) *reinterpret_cast<floatx4*>(piece + (4 * r + r0) * 64 + 4 * (chunk ^ ((4 * r + r0) & 15))) = st.x[r];
      __builtin_amdgcn_wave_barrier();
      if (ft + 1 < DT) load_k(full, ft + 1);
      else load_v(full, 0);
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const floatx4 kx = *reinterpret_cast<const floatx4*>(piece + lane * 64 + 4 * (c ^ (lane & 15)));
        s0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kx[0], q[ft][4 * c + 0], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_4x4x1f32(kx[1], q[ft][4 * c + 1], s1, 0, 0, 0);
        s0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kx[2], q[ft][4 * c + 2], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_4x4x1f32(kx[3], q[ft][4 * c + 3], s1, 0, 0, 0);
      }
    }
    // softmax: this lane has head lane % 4 of keys 4 (lane / 4) .. + 3
    const int v0 = t * 64 + (lane & ~3);
    float s[4], tmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = v0 + i < total ? (flat ? 0.f : (s0[i] + s1[i]) * A.scale) : -INFINITY;
      tmax = fmaxf(tmax, s[i]);
    }
    const float mn = fmaxf(S.m, max_mod4(tmax)), mref = mn == -INFINITY ? 0.f : mn;      // (keys whose scores overflow to -inf weigh nothing)
    const float alpha = expf(S.m - mref);              // m = -inf: 0
    S.m = mn;
    float p[4], ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) { p[i] = expf(s[i] - mref); ps += p[i]; }
    S.l = S.l * alpha + ps;
    floatx4 al;
#pragma unroll
    for (int h = 0; h < 4; ++h) al[h] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, alpha), h));
#pragma unroll
    for (int ft = 0; ft < DT; ++ft) {
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (FULL || r < 4 || r / 4 < here) *reinterpret_cast<floatx4*>(piece + (4 * r + r0) * 64 + 4 * chunk) = st.x[r];
      __builtin_amdgcn_wave_barrier();
      if (ft + 1 < DT) load_v(full, ft + 1);
      else if (t + step < tiles) {
        locate(t + step);
        quarters = quarters_of(t + step);
        if (DT > 1 || quarters == 4) load_k(Full{}, 0);
        else load_k(Part{}, 0);
      }
      floatx4 o0 = S.acc[ft] * al, o1 = {0.f, 0.f, 0.f, 0.f};
      static_for<0, 4>([&](auto quarter) {
        constexpr int qd = decltype(quarter)::value;
        if (FULL || qd == 0 || qd < here)
          static_for<4 * qd, 4 * qd + 4>([&](auto blk) {
            constexpr int b = decltype(blk)::value;
            const float* vr = piece + 4 * b * 64 + lane;
            o0 = __builtin_amdgcn_mfma_f32_4x4x1f32(p[0], vr[0], o0, 4, b, 0);
            o1 = __builtin_amdgcn_mfma_f32_4x4x1f32(p[1], vr[64], o1, 4, b, 0);
            o0 = __builtin_amdgcn_mfma_f32_4x4x1f32(p[2], vr[128], o0, 4, b, 0);
            o1 = __builtin_amdgcn_mfma_f32_4x4x1f32(p[3], vr[192], o1, 4, b, 0);
          });
      });
      S.acc[ft] = o0 + o1;
    }
  };
  for (int t = first; t < tiles; t += step) {
    if (DT > 1 || quarters == 4) tile(Full{}, t);
    else tile(Part{}, t);
  }
}

// SELECT: block selection, else interval masks.  WPQ: waves of a work-group that share a query (1 or 4; with 4 each takes
// every fourth tile and the partial results are merged: few queries, long key lists).
struct RowsShared {
  float pieces[4 * kRowsPiece];
  int blocks[4][64], rows[4][64];
};

template <int DT, bool SELECT, int WPQ>
__device__ __forceinline__ void f32_rows_body(const F32Args& A, const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                                              const void* __restrict__ idx, const uint8_t* __restrict__ fmask, float* __restrict__ out,
                                              float* __restrict__ lse, RowsShared& sh) {
  float* pieces = sh.pieces;
  int (&blocks_s)[4][64] = sh.blocks;
  int (&rows_s)[4][64] = sh.rows;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = WPQ == 1 ? blockIdx.x * 4 + wave : blockIdx.x;
  if (i >= A.n) return;                                   // (WPQ == 1: no work-group barrier follows)
  const int bh = blockIdx.y, b = bh / A.hk, hk = bh % A.hk;
  const float* kb = k + b * A.sk[0] + hk * A.sk[1];
  const float* vb = v + b * A.sv[0] + hk * A.sv[1];
  float* piece = pieces + wave * kRowsPiece;
  int* blocks = blocks_s[wave];
  const int first = WPQ == 1 ? 0 : wave, step = WPQ;
  const int pos = i + A.qoff;
  const float* mk = A.memk != nullptr ? A.memk + (long)hk * A.mem * A.d : kb;
  const float* mv = A.memv != nullptr ? A.memv + (long)hk * A.mem * A.d : vb;
  // A query of a non-causal selection whose slots are all dead attends their blocks uniformly, zero padding included: the
  // reference fills all its logits with the same value (NSA.py:809-815).
  bool dead = false;
  if constexpr (SELECT) {
    if (A.uniform) {
      dead = true;
      for (int s = lane; s < A.S; s += 64)
        if (fmask[((size_t)bh * A.n + i) * A.S + s]) dead = false;      // (a live slot that names no block: nothing attended, as before)
      dead = !__any(!dead);
    }
  }
  for (int g0 = 0; g0 < A.g; g0 += 4) {
    float qr[DT][64];
    {
      // (heads past the group repeat its last one and are not stored; features past the head dimension meet zero keys)
      const int g = min(g0 + (lane & 3), A.g - 1);
      int last = A.d - 1;
      asm volatile("" : "+s"(last));          // (the 64 clamped offsets are not worth registers across the loop over heads)
      const float* qp = q + b * A.sq[0] + (long)(hk * A.g + g) * A.sq[1] + (long)i * A.sq[2];
#pragma unroll
      for (int ft = 0; ft < DT; ++ft)
#pragma unroll
        for (int e = 0; e < 64; ++e) qr[ft][e] = qp[min(64 * ft + e, last)];
    }
    RowsState<DT> S;
    S.m = -INFINITY;
    S.l = 0.f;
#pragma unroll
    for (int ft = 0; ft < DT; ++ft) S.acc[ft] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (SELECT) {
      // the live slots' blocks one after the other, 64 slots at a time, and behind the last the own block up to the query
      const int own = A.causal ? pos / A.B : 0, own_keys = A.causal ? pos - own * A.B + 1 : 0;
      int s0 = 0;
      do {
        int blk = -1;
        if (s0 + lane < A.S) {
          const size_t at = ((size_t)bh * A.n + i) * A.S + s0 + lane;
          if (dead || fmask[at]) {
            const long j = A.idx64 ? (long)reinterpret_cast<const long long*>(idx)[at] : (long)reinterpret_cast<const int*>(idx)[at];
            if (dead) blk = (int)min(max(j, 0l), (long)A.W - 1);
            else if (j >= 0 && j < A.W) blk = (int)j;
          }
        }
        const unsigned long long live = __ballot(blk >= 0);
        const int cnt = __popcll(live);
        __builtin_amdgcn_wave_barrier();
        if (blk >= 0) blocks[__popcll(live & ((1ull << lane) - 1))] = blk;
        __builtin_amdgcn_wave_barrier();
        const bool last = s0 + 64 >= A.S;
        rows_walk<DT>(A, piece, rows_s[wave], qr, kb, vb, kb, vb, cnt * A.B + (last ? own_keys : 0), first, step, dead, [&](int v) {
          const int slot = v / A.B, off = v - slot * A.B;
          const int row = (slot < cnt ? blocks[slot] : own) * A.B + off;
          return row < A.nk ? row : -1;
        }, S, lane);
        s0 += 64;
      } while (s0 < A.S);
    } else {
      int lo, hi;
      f32_interval(A, pos, lo, hi);
      const int own_mem = A.memk != nullptr ? A.mem : 0;
      rows_walk<DT>(A, piece, rows_s[wave], qr, kb, vb, mk, mv, hi - lo + 1, first, step, false, [&](int v) {
        const int u = lo + v;
        return u < own_mem ? -2 - u : u - own_mem;
      }, S, lane);
    }
    float l = sum_mod4(S.l);
    float* ob = out + (((long)b * A.hk * A.g + (long)hk * A.g + g0) * A.n + i) * A.d;
    if constexpr (WPQ == 1) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        if (g0 + h >= A.g) break;
        const float lh = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, l), h));
        const float inv = lh > 0.f ? 1.0f / lh : 0.f;
#pragma unroll
        for (int ft = 0; ft < DT; ++ft)
          if (64 * ft + lane < A.d) ob[(long)h * A.n * A.d + 64 * ft + lane] = S.acc[ft][h] * inv;
      }
      if (lse != nullptr && lane < 4 && g0 + lane < A.g)
        lse[((long)b * A.hk * A.g + (long)hk * A.g + g0 + lane) * A.n + i] = l > 0.f && !dead ? S.m + logf(l) : -INFINITY;
    } else {
      // merge of the four waves' partial results: wave w finishes head g0 + w
      __syncthreads();                                     // the pieces are free
      float* part = pieces;                                // [wave][head]: m, l, features
      if (lane < 4) { part[(wave * 4 + lane) * (2 + 64 * DT)] = S.m; part[(wave * 4 + lane) * (2 + 64 * DT) + 1] = l; }
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int ft = 0; ft < DT; ++ft) part[(wave * 4 + h) * (2 + 64 * DT) + 2 + 64 * ft + lane] = S.acc[ft][h];
      __syncthreads();
      if (g0 + wave < A.g) {
        float mm = -INFINITY, ll = 0.f, o[DT];
#pragma unroll
        for (int w = 0; w < 4; ++w) mm = fmaxf(mm, part[(w * 4 + wave) * (2 + 64 * DT)]);
#pragma unroll
        for (int ft = 0; ft < DT; ++ft) o[ft] = 0.f;
        const float mref = mm == -INFINITY ? 0.f : mm;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float* pw = part + (w * 4 + wave) * (2 + 64 * DT);
          const float a = expf(pw[0] - mref);              // a wave without a tile: m = -inf, weight 0
          ll += pw[1] * a;
#pragma unroll
          for (int ft = 0; ft < DT; ++ft) o[ft] += pw[2 + 64 * ft + lane] * a;
        }
        const float inv = ll > 0.f ? 1.0f / ll : 0.f;
#pragma unroll
        for (int ft = 0; ft < DT; ++ft)
          if (64 * ft + lane < A.d) ob[(long)wave * A.n * A.d + 64 * ft + lane] = o[ft] * inv;
        if (lse != nullptr && lane == 0)
          lse[((long)b * A.hk * A.g + (long)hk * A.g + g0 + wave) * A.n + i] = ll > 0.f && !dead ? mm + logf(ll) : -INFINITY;
      }
      __syncthreads();                                     // before the next heads' pieces overwrite the partials
    }
  }
}

template <int DT, bool SELECT, int WPQ>
__global__ __launch_bounds__(256, 2) void f32_rows_kernel(const F32Args A, const float* __restrict__ q, const float* __restrict__ k,
                                                          const float* __restrict__ v, const void* __restrict__ idx,
                                                          const uint8_t* __restrict__ fmask, float* __restrict__ out, float* __restrict__ lse) {
  __shared__ RowsShared sh;
  f32_rows_body<DT, SELECT, WPQ>(A, q, k, v, idx, fmask, out, lse, sh);
}

// Two interval masks of as many queries in one launch (the compressed branch and the window of a few tokens: a launch each is
// most of their time)
struct RowsCall { F32Args A; const float *q, *k, *v; float* out; };

template <int DT, int WPQ>
__global__ __launch_bounds__(256, 2) void f32_rows_pair_kernel(const RowsCall X, const RowsCall Y) {
  __shared__ RowsShared sh;
  if (blockIdx.z == 0) f32_rows_body<DT, false, WPQ>(X.A, X.q, X.k, X.v, nullptr, nullptr, X.out, nullptr, sh);
  else f32_rows_body<DT, false, WPQ>(Y.A, Y.q, Y.k, Y.v, nullptr, nullptr, Y.out, nullptr, sh);
}

// ------------------------------------------------------------------------------------------ tile
//
// Many queries: a wave holds 32 rows (row r of a kv head = query r / G, head r % G, so any group size fits), a work-group 128;
// tiles of 32 keys of K and V are shared through LDS, double-buffered, one barrier per tile.  The products are made of bf16
// thirds (nsa_split.hpp): K and V are split on their way into LDS, once for the 128 rows, Q once and P where it is made.
//   S^T = K Q^T: A = K (lane = key), B = Q (lane = row);  O^T = V^T P^T: A = V^T by the LDS transpose load, whose order of rows is the
//   order in which S^T's registers hold the keys, so P goes in as it is.
// Interval masks, and (SEL) block selections of few enough blocks: every tile of a block that one of the 128 rows selected is
// multiplied and a row's own choice is a mask on the scores, which beats gathering while a query attends a fair share of the
// blocks there are (f32_masked_tiles).
// Per tile and wave at d = 64 64 MFMAs (2048 cycles) and some 450 vector instructions (the split of K, V and P 230, softmax 160),
// of which two waves to a SIMD hide part of each other; a wave alone takes 2.6 us.  Against v_mfma_f32_32x32x2 tiles (64 MFMAs of 64
// cycles): 2 x 2053 queries, 16 heads x 4 kv heads, window 512 110 -> 72 us, strided prefix 34 -> 28; 32 x 8 heads, d = 128, 2000 queries
// 181 -> 155.  Error of the outputs against float64, rms: window 512 3.9e-8 -> 1.6e-8, two keys 6.6e-8 -> 4.6e-8.
constexpr int kTileBlocks = 128;         // blocks of a masked selection

// Which tile of 128 rows of which (batch, kv head) pair a work-group takes.  Longest key lists first (causal prefixes).  Where the
// launch fits the chip at two work-groups to a CU, the second half goes the other way round: the longest then shares its CU with the
// shortest (1 x 4096 queries, 16 heads x 4 kv heads, d = 64: window of all 268 -> 258 us, strided prefix 27.9 -> 27.2, masked
// selection 296 -> 291).  At d = 128 a CU holds one, and the second half starts where the first ends: longest first there, too (1 x
// 2000 queries, 32 x 8 heads, turned 300 us, not 242).  The ids are turned, not the tiles: a pair's tiles may lie on both sides of id 256.
struct TilePlace { int pair, tile; };
__host__ __device__ inline TilePlace f32_tile_place(int id, int grid, int pairs, bool two_to_a_cu) {
  if (two_to_a_cu && grid <= 512 && id >= 256) id = 255 + grid - id;
  return TilePlace{id % pairs, grid / pairs - 1 - id / pairs};
}

__device__ __forceinline__ void split_probs(const float (&p)[16], bf16x8 (&part)[3][2]) {
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    uint32_t w[3][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t s[3];
      split2(p[8 * u + 2 * j], p[8 * u + 2 * j + 1], s);
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) w[pl][j] = s[pl];
    }
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) part[pl][u] = __builtin_bit_cast(bf16x8, uintx4{w[pl][0], w[pl][1], w[pl][2], w[pl][3]});
  }
}

template <int D, bool SEL>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void f32_tile_kernel(const F32Args A, const float* __restrict__ q, const float* __restrict__ k,
                                                                        const float* __restrict__ v, const void* __restrict__ idx,
                                                                        const uint8_t* __restrict__ fmask, float* __restrict__ out,
                                                                        float* __restrict__ lse) {
  constexpr int KP = D + 8, VP = D + 16;                 // row strides: conflict-free row reads of K, transpose loads of V
  constexpr int LD = D / 32, KS = D / 16, FT = D / 32;
  __shared__ __align__(16) __bf16 k_s[2][3 * 32 * KP];
  __shared__ __align__(16) __bf16 v_s[2][3 * 32 * VP];   // (zeros for values that are not finite)
  __shared__ int odd_s;                                  // there was such a value
  __shared__ uint32_t mask_s[SEL ? 129 : 1][kTileBlocks / 32], any_s[kTileBlocks / 32];
  __shared__ int repeated_s, big_s;                      // big_s: some key was that large (it stays set)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n_ = lane & 31, h = lane >> 5;
  const TilePlace at = f32_tile_place(blockIdx.x, gridDim.x, A.bh, D == 64);
  const int b = at.pair / A.hk, hk = at.pair % A.hk;
  const float* kb = k + b * A.sk[0] + hk * A.sk[1];
  const float* vb = v + b * A.sv[0] + hk * A.sv[1];
  const long all_rows = (long)A.n * A.g;
  const long row0 = (long)at.tile * 128;
  const long row = row0 + wave * 32 + n_;
  const long rowc = row < all_rows ? row : all_rows - 1;
  const int qi = (int)(rowc / A.g), g = (int)(rowc - (long)qi * A.g);
  const int gq0 = (int)(row0 / A.g), gq1 = (int)(min(row0 + 127, all_rows - 1) / A.g);
  // Keys [lo, lo + seen] are visible to the row, and (SEL) those of its selected blocks.
  // g_lo .. g_hi: what the work-group walks; w_lo .. w_hi: what the wave's rows see of the interval.
  int lo, hi, w_lo, w_hi, g_lo, g_hi, dummy;
  const int wq0 = (int)(min(row0 + wave * 32, all_rows - 1) / A.g), wq1 = (int)(min(row0 + wave * 32 + 31, all_rows - 1) / A.g);
  if (SEL) {
    hi = qi + A.qoff;
    lo = (hi >> A.lb) << A.lb;
    w_lo = ((wq0 + A.qoff) >> A.lb) << A.lb;
    w_hi = wq1 + A.qoff;
    g_lo = 0;
    g_hi = gq1 + A.qoff;
  } else {
    f32_interval(A, qi + A.qoff, lo, hi);
    f32_interval(A, wq0 + A.qoff, w_lo, dummy);
    f32_interval(A, wq1 + A.qoff, dummy, w_hi);
    f32_interval(A, gq0 + A.qoff, g_lo, dummy);
    f32_interval(A, gq1 + A.qoff, dummy, g_hi);
    if (A.mode == 1) { w_hi = max(w_hi, A.mem - 1); g_hi = max(g_hi, A.mem - 1); hi = max(hi, A.mem - 1); }
  }
  // a key is visible if key - lo, as an unsigned number, is at most `seen`: one comparison, and no branch per element
  const unsigned seen = hi < lo ? 0u : (unsigned)(hi - lo);
  if (hi < lo) lo = 0x7fffffff;

  unsigned long long any0 = 0, any1 = 0;                 // blocks that some row of the work-group attends
  bool repeated = false;
  const size_t slot0 = SEL ? ((size_t)at.pair * A.n + gq0) * A.S : 0;
  auto block_of = [&](size_t at) {
    if (!fmask[at]) return -1;
    const long j = A.idx64 ? (long)reinterpret_cast<const long long*>(idx)[at] : (long)reinterpret_cast<const int*>(idx)[at];
    return j >= 0 && j < A.W ? (int)j : -1;
  };
  if (SEL) {
    for (int e = tid; e < 129 * (kTileBlocks / 32); e += 256) (&mask_s[0][0])[e] = 0;
    if (tid < kTileBlocks / 32) any_s[tid] = 0;
    if (tid == 0) repeated_s = 0;
    __syncthreads();
    const int total = (gq1 - gq0 + 1) * A.S;
    for (int e = tid; e < total; e += 256) {
      const int j = block_of(slot0 + e);
      if (j < 0) continue;
      const int qr = e / A.S;
      const uint32_t bit = 1u << (j & 31);
      // a block named twice, or the own block or a later one: the masks cannot say that (the scores' weights can, below)
      if ((atomicOr(&mask_s[qr][j >> 5], bit) & bit) || j >= (gq0 + qr + A.qoff) >> A.lb) repeated_s = 1;
      atomicOr(&any_s[j >> 5], bit);
    }
    for (int qr = tid; qr <= gq1 - gq0; qr += 256) {
      const int own = (gq0 + qr + A.qoff) >> A.lb;
      atomicOr(&any_s[own >> 5], 1u << (own & 31));
    }
    __syncthreads();
    auto word = [&](int w) { return (unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)any_s[w]); };
    any0 = word(0) | word(1) << 32;
    any1 = word(2) | word(3) << 32;
    repeated = __builtin_amdgcn_readfirstlane(repeated_s) != 0;
    if (repeated) g_hi = (A.W << A.lb) - 1;              // (zero padding behind the last key counts, as a score of 0)
  }
  // the first tile from t0 on that somebody attends
  const uint32_t tile_bits = SEL ? (1u << max(1, 32 >> A.lb)) - 1u : 0;
  auto attended = [&](int t0) {
    if (SEL) {
      while (t0 <= g_hi) {
        const int j = t0 >> A.lb;
        if (((j < 64 ? any0 >> j : any1 >> (j - 64)) & tile_bits) != 0) break;
        t0 += 32;
      }
    }
    return t0;
  };

  // Products of numbers below kBig do not overflow; where larger ones (or infinities) meet, a sum of leading products may not be
  // finite, and the small ones then mean nothing.
  constexpr float kBig = 1.152921504606846976e18f;       // 2^60
  bool q_big;
  bf16x8 qf[3][KS];
  {
    // (a negative scale goes into the queries, so that the largest product is the largest score)
    const float sign = A.scale < 0.f ? -1.f : 1.f;
    const float* qp = q + b * A.sq[0] + (long)(hk * A.g + g) * A.sq[1] + (long)qi * A.sq[2];
    float big = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint32_t w[3][4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int f = 16 * ks + 8 * h + 2 * j;
        const float x0 = qp[min(f, A.d - 1)], x1 = qp[min(f + 1, A.d - 1)];
        big = fmaxf(big, fmaxf(fabsf(x0), fabsf(x1)));
        uint32_t s[3];
        split2(f < A.d ? sign * x0 : 0.f, f + 1 < A.d ? sign * x1 : 0.f, s);
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) w[pl][j] = s[pl];
      }
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) qf[pl][ks] = __builtin_bit_cast(bf16x8, uintx4{w[pl][0], w[pl][1], w[pl][2], w[pl][3]});
    }
    q_big = __any(big >= kBig);
  }
  floatx16 o[FT], os[FT];                                // sums of leading and of small products
#pragma unroll
  for (int ft = 0; ft < FT; ++ft) { o[ft] = zero_acc(); os[ft] = zero_acc(); }
  // Weights are powers of two of (score - maximum) (c + c_lo), scale x log2 e in two parts: the rounding of c alone would change every
  // weight of a row the same way.  c is cut off, so that c_lo is positive and a score of minus infinity stays one (a scale of 0 as well).
  const float scale = fabsf(A.scale), c = fmaxf(scale * kLog2e * (1.f - 0x1p-22f), 1e-37f);
  const float c_lo = fmaxf(__builtin_fmaf(scale, kLog2e, -c) + scale * 1.925963e-8f, 2e-38f);
  auto weight = [&](float below) { return fast_exp2(__builtin_fmaf(below, c_lo, below * c)); };
  float m = -INFINITY, l = 0.f;                          // m: of the unscaled scores

  const int own_mem = A.memk != nullptr ? A.mem : 0;
  const int last_key = SEL ? min(g_hi, A.nk - 1) : g_hi;
  floatx4 kx[LD], vx[LD];
  // this thread's rows of a tile that lies within the keys: offsets from its first row (row strides: below 2^24)
  unsigned k_at[LD], v_at[LD];
#pragma unroll
  for (int u = 0; u < LD; ++u) {
    const int e = u * 256 + tid, r = e / (D / 4), ch = e % (D / 4);
    k_at[u] = (unsigned)r * (unsigned)A.sk[2] + 4 * ch;
    v_at[u] = (unsigned)r * (unsigned)A.sv[2] + 4 * ch;
  }
  const bool plain_rows = A.d == D && A.sk[2] >= 0 && A.sv[2] >= 0 && (A.sk[2] | A.sv[2]) >> 24 == 0;
  auto fetch = [&](int t0) {
    if (plain_rows && t0 >= own_mem && t0 + 31 <= last_key) {
      const float *kt = kb + (long)(t0 - own_mem) * A.sk[2], *vt = vb + (long)(t0 - own_mem) * A.sv[2];
#pragma unroll
      for (int u = 0; u < LD; ++u) {
        kx[u] = *reinterpret_cast<const floatx4*>(kt + k_at[u]);
        vx[u] = *reinterpret_cast<const floatx4*>(vt + v_at[u]);
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < LD; ++u) {
      const int e = u * 256 + tid, r = e / (D / 4), ch = e % (D / 4);
      const int kr = t0 + r;
      floatx4 z = {0.f, 0.f, 0.f, 0.f};
      kx[u] = z;
      vx[u] = z;
      if (kr <= last_key && 4 * ch < A.d) {
        const bool own = kr < own_mem;
        kx[u] = *reinterpret_cast<const floatx4*>((own ? A.memk + ((long)hk * A.mem + kr) * A.d : kb + (long)(kr - own_mem) * A.sk[2]) + 4 * ch);
        vx[u] = *reinterpret_cast<const floatx4*>((own ? A.memv + ((long)hk * A.mem + kr) * A.d : vb + (long)(kr - own_mem) * A.sv[2]) + 4 * ch);
      }
    }
  };
  int t0 = attended(g_lo & ~31);
  fetch(t0);
  if (tid == 0) { odd_s = 0; big_s = 0; }
  __syncthreads();
  bool odd = false;
  int buf = 0;
  for (; t0 <= g_hi; buf ^= 1) {
    bool k_big = false;
    float zero = 0.f;
#pragma unroll
    for (int u = 0; u < LD; ++u) {
      k_big |= fmaxf(fmaxf(fabsf(kx[u][0]), fabsf(kx[u][1])), fmaxf(fabsf(kx[u][2]), fabsf(kx[u][3]))) >= kBig;
#pragma unroll
      for (int e = 0; e < 4; ++e) zero = __builtin_fmaf(vx[u][e], 0.f, zero);      // (NaN if one of them is not finite)
    }
    if (__any(zero != 0.f)) {
      odd = true;
#pragma unroll
      for (int u = 0; u < LD; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) vx[u][e] = fabsf(vx[u][e]) < INFINITY ? vx[u][e] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < LD; ++u) {
      const int e = u * 256 + tid, r = e / (D / 4), ch = e % (D / 4);
      const Split3 ks = split4(kx[u]), vs = split4(vx[u]);
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) {
        *reinterpret_cast<bf16x4*>(&k_s[buf][(pl * 32 + r) * KP + 4 * ch]) = ks.part[pl];
        *reinterpret_cast<bf16x4*>(&v_s[buf][(pl * 32 + r) * VP + 4 * ch]) = vs.part[pl];
      }
    }
    if (k_big) big_s = 1;
    __syncthreads();          // (the other buffer was read before this barrier by every wave: it may be written in the next round)
    const int here = t0;
    t0 = attended(t0 + 32);
    if (t0 <= g_hi) fetch(t0);
    uint32_t chosen = 0;      // bit i: the row selected block i of the tile
    if (SEL) {
      const int j = here >> A.lb;
      chosen = (mask_s[qi - gq0][j >> 5] >> (j & 31)) & tile_bits;
      if (!__any(chosen != 0) && (here > w_hi || here + 31 < w_lo)) continue;
    } else if (here > w_hi || here + 31 < w_lo) {
      continue;               // wave-uniform: nothing of this tile is visible to the wave
    }
    const int overflows = big_s;
    floatx16 lead = zero_acc(), small = zero_acc();
    // (operands are read a product group ahead: at one or two waves per SIMD an LDS round trip in front of every group is not hidden)
    bf16x8 kf[2][3], vf[2][3];
    auto read_k = [&](int ks) {
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) kf[ks & 1][pl] = *reinterpret_cast<const bf16x8*>(&k_s[buf][(pl * 32 + n_) * KP + 16 * ks + 8 * h]);
    };
    auto read_v = [&](int g) {                            // group g: keys 16 (g / FT), features 32 (g % FT)
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) vf[g & 1][pl] = lds_transposed_operand(&v_s[buf][pl * 32 * VP], VP, 16 * (g / FT), 32 * (g % FT), lane);
    };
    read_k(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 1 < KS) read_k(ks + 1);
      const bf16x8 (&kk)[3] = kf[ks & 1];
      lead = mfma32(kk[0], qf[0][ks], lead);
      small = mfma32(kk[0], qf[1][ks], small);
      small = mfma32(kk[0], qf[2][ks], small);
      small = mfma32(kk[1], qf[0][ks], small);
      small = mfma32(kk[1], qf[1][ks], small);
      small = mfma32(kk[1], qf[2][ks], small);
      small = mfma32(kk[2], qf[0][ks], small);
      small = mfma32(kk[2], qf[1][ks], small);
    }
    read_v(0);
    if (q_big || __builtin_amdgcn_readfirstlane(overflows)) {
#pragma unroll
      for (int i = 0; i < 16; ++i) small[i] = fabsf(lead[i]) < INFINITY ? small[i] : 0.f;
    }
    float sv[16], tmax = -INFINITY;
    const int from_lo = here + 4 * h - lo;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const unsigned limit = SEL && ((chosen >> ((8 * a + 4 * h) >> A.lb)) & 1u) ? 0xffffffffu : seen;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * a + e;
        sv[i] = (unsigned)(from_lo + 8 * a + e) <= limit ? lead[i] + small[i] : -INFINITY;
        tmax = fmaxf(tmax, sv[i]);
      }
    }
    tmax = halves_max(tmax);
    // (a reference that lags behind the maximum would spare most tiles the multiplication of the sums, 1 to 4 % of the time, but weights
    // above 1 carry large values over the end of fp32, and the lse of 512 keys was 3.4e-7 off in the mean, not 2.8e-7)
    const float mn = fmaxf(m, tmax), mref = mn == -INFINITY ? 0.f : mn;
    const float alpha = weight(m - mref);                // m = -inf: 0
    m = mn;
    float ps = 0.f;
    if (SEL && repeated) {
      // weights: how often the row's live slots name a key's block, and once more where the key is the own block's
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int j = (here + 8 * a + 4 * h) >> A.lb;
        int times = 0;
        for (int s = 0; s < A.S; ++s) times += block_of(slot0 + (size_t)(qi - gq0) * A.S + s) == j;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float w = (float)(times + ((unsigned)(from_lo + 8 * a + e) <= seen ? 1 : 0));
          sv[4 * a + e] = w > 0.f ? w * weight(sv[4 * a + e] - mref) : 0.f;
          ps += sv[4 * a + e];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) { sv[i] = weight(sv[i] - mref); ps += sv[i]; }
    }
    l = l * alpha + ps;                                  // this half's keys
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int ft = 0; ft < FT; ++ft)
#pragma unroll
        for (int i = 0; i < 16; ++i) { o[ft][i] *= alpha; os[ft][i] *= alpha; }
    }
    bf16x8 pf[3][2];
    split_probs(sv, pf);
#pragma unroll
    for (int gr = 0; gr < 2 * FT; ++gr) {
      if (gr + 1 < 2 * FT) read_v(gr + 1);
      const bf16x8 (&vv)[3] = vf[gr & 1];
      const int u = gr / FT, ft = gr % FT;
      o[ft] = mfma32(vv[0], pf[0][u], o[ft]);
      os[ft] = mfma32(vv[0], pf[1][u], os[ft]);
      os[ft] = mfma32(vv[0], pf[2][u], os[ft]);
      os[ft] = mfma32(vv[1], pf[0][u], os[ft]);
      os[ft] = mfma32(vv[1], pf[1][u], os[ft]);
      os[ft] = mfma32(vv[1], pf[2][u], os[ft]);
      os[ft] = mfma32(vv[2], pf[0][u], os[ft]);
      os[ft] = mfma32(vv[2], pf[1][u], os[ft]);
    }
  }
  // A value that is not finite is left out of the products, where a weight of zero times it would be NaN in every row of its tile,
  // and added here to the rows that see its key.
  if (odd) odd_s = 1;
#pragma unroll
  for (int ft = 0; ft < FT; ++ft)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[ft][i] += os[ft][i];
  __syncthreads();
  if (odd_s) {
#pragma unroll 1
    for (int kr = g_lo; kr <= last_key; ++kr) {
      const float* vr = kr < own_mem ? A.memv + ((long)hk * A.mem + kr) * A.d : vb + (long)(kr - own_mem) * A.sv[2];
      bool visible = (unsigned)(kr - lo) <= seen;
      if (SEL) visible |= (mask_s[qi - gq0][(kr >> A.lb) >> 5] >> ((kr >> A.lb) & 31)) & 1u;
#pragma unroll
      for (int ft = 0; ft < FT; ++ft)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int f0 = 32 * ft + 8 * u + 4 * h;
          if (f0 >= A.d) continue;
          const floatx4 x = *reinterpret_cast<const floatx4*>(vr + f0);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (visible && !(fabsf(x[e]) < INFINITY)) o[ft][4 * u + e] += x[e];
        }
    }
  }
  l = halves_sum(l);
  if (row >= all_rows) return;
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  const long orow = ((long)b * A.hk * A.g + (long)hk * A.g + g) * A.n + qi;
  float* op = out + orow * A.d;
#pragma unroll
  for (int ft = 0; ft < FT; ++ft)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int f0 = 32 * ft + 8 * u + 4 * h;
      if (f0 < A.d)
        *reinterpret_cast<floatx4*>(op + f0) = floatx4{o[ft][4 * u] * inv, o[ft][4 * u + 1] * inv, o[ft][4 * u + 2] * inv, o[ft][4 * u + 3] * inv};
    }
  if (lse != nullptr && h == 0) lse[orow] = l > 0.f ? __builtin_fmaf(m, fabsf(A.scale), logf(l)) : -INFINITY;
}

static int f32_common(int batch, int kv_heads, int group, int seq, int q_offset, int dim_head, float scale, const int64_t* qs, const int64_t* ks,
                      const int64_t* vs, F32Args& A) {
  if (batch <= 0 || kv_heads <= 0 || group <= 0 || seq <= 0 || q_offset < 0) return NSA_E_ARG;
  A.qoff = q_offset;
  if (dim_head <= 0 || dim_head > kF32MaxD || (dim_head & 3)) return NSA_E_UNSUPPORTED;
  if ((long)batch * kv_heads > 65535) return NSA_E_UNSUPPORTED;
  A.b = batch; A.hk = kv_heads; A.bh = batch * kv_heads; A.g = group; A.n = seq; A.d = dim_head; A.scale = scale;
  for (int t = 0; t < 3; ++t) {
    A.sq[t] = qs[t]; A.sk[t] = ks[t]; A.sv[t] = vs[t];
    if ((A.sk[t] | A.sv[t]) & 3) return NSA_E_ARG;       // key / value rows are read 16 bytes at a time
  }
  return 0;
}

// A query per wave once the queries fill the chip, else a query per work-group (its four waves share the keys).  Measured at
// 17 blocks of 64 keys, d = 64: 1024 queries 52 us shared, 55 us one per wave; 2048 queries 95 against 82 us.  Interval masks
// have shorter key lists (down to one tile): 1024 queries, window 512, 22 us either way, 2048 queries 48 against 41 us.
template <bool SELECT>
static void f32_launch_rows(const F32Args& A, const float* q, const float* k, const float* v, const void* idx, const uint8_t* fmask, float* out,
                            float* lse, hipStream_t stream) {
  const long queries = (long)A.n * A.b * A.hk;
  const bool shared = queries < (SELECT ? 2048 : 1024);
  const dim3 grid(shared ? A.n : (A.n + 3) / 4, A.b * A.hk);
#define NSA_ROWS(DT, WPQ) hipLaunchKernelGGL((f32_rows_kernel<DT, SELECT, WPQ>), grid, dim3(256), 0, stream, A, q, k, v, idx, fmask, out, lse)
  if (A.d <= 64) { if (shared) NSA_ROWS(1, 4); else NSA_ROWS(1, 1); }
  else { if (shared) NSA_ROWS(2, 4); else NSA_ROWS(2, 1); }
#undef NSA_ROWS
}

template <bool SEL>
static void f32_launch_tiles(const F32Args& A, const float* q, const float* k, const float* v, const void* idx, const uint8_t* fmask, float* out,
                             float* lse, hipStream_t stream) {
  const dim3 grid((unsigned)((((long)A.n * A.g + 127) / 128) * A.bh));
  if (A.d <= 64) hipLaunchKernelGGL((f32_tile_kernel<64, SEL>), grid, dim3(256), 0, stream, A, q, k, v, idx, fmask, out, lse);
  else hipLaunchKernelGGL((f32_tile_kernel<128, SEL>), grid, dim3(256), 0, stream, A, q, k, v, idx, fmask, out, lse);
}

// A work-group of the tile kernel needs some 128 rows, and the launch enough of them.  Interval masks, us row by row / in tiles:
//   d = 64   2048 queries, 16 / 4 heads 38 / 42 (window 512), 12.8 / 14.6 (64); 4096 76 / 45 and 22 / 16; 3072 59 / 44 and 21 / 15, window 2 12 / 13;
//            8 / 8 heads 2048 20.5 / 24.7 and 10.6 / 20.4, 4096 56 / 41 and 19 / 20.5
//   d = 128  32 / 8 heads 512 queries 21 / 21, 768 40 / 25, 1024 27.6 / 27.7 (window 512), 20 / 21 (2); 2048 58 / 42 and 28 / 21
//            narrow windows of groups of 1 and 2, 1024 to 2048 queries: 8 / 8 heads, 1024 18 / 28 (2 to 32), 26 / 28 (64), 2048 22 / 32 (2), 26 / 32 (32), 34 / 36
//            (64); 16 / 8 heads, 1024 20 / 25 (2 to 32); but 768 31 / 23 (2), 3200 40 / 32 (2)
static bool f32_tiles_fit(const F32Args& A) {
  const long queries = (long)A.n * A.b * A.hk;
  if ((long)A.n * A.g < 128 || queries < (A.d <= 64 ? 4096 : 512)) return false;
  const bool narrow = A.B == 0 && A.mode == 0 && A.g <= 2 && A.wb < 48 && A.wf < 48;      // (a window, not a selection)
  return !(A.d > 64 && narrow && queries >= 1024 && queries <= 2048);
}

// Masked tiles instead of gathered blocks, where the blocks fit the masks and the estimate of the time (us) is lower:
//   tiles   a work-group's walk to the last key, 2.5 us per 32 keys (d = 128: 5), or the chip's rate over all rows and half the keys
//   gather  per query (four heads at a time) 1.4 ns (4.6) for 64 keys of its blocks + 3 (12)
// Measured, gather / tiles: 16 blocks of 64, d = 64, G 4: 2 x 2053 queries x 4 451 / 183, 1024 x 4 99 / 85, 8192 x 4 979 / 882; 4 blocks of 64, G 1 4000 x 8
// 328 / 306; 4 blocks of 16, G 2: 8 x 1024 x 4 154 / 90, 4 x 1024 x 4 82 / 86, 2 x 1024 x 4 45 / 85, 4 x 2048 x 4 157 / 165; d = 128, 16 of 64: 2048 x 8 1301 / 314;
// 4 of 16: 2048 x 8 297 / 298; 4 of 64: 8192 x 8 2351 / 3381.
static bool f32_masked_tiles(F32Args& A) {
  A.lb = 0;
  while (A.lb < 30 && (1 << A.lb) < A.B) ++A.lb;
  if (!A.causal || A.B < 4 || A.B != 1 << A.lb || A.W > kTileBlocks || !f32_tiles_fit(A)) return false;
  const bool wide = A.d > 64;
  const double queries = (double)A.n * A.b * A.hk, keys = (double)(A.S + 1) * A.B;
  const double tiles = std::max(A.nk * (wide ? 0.16 : 0.079), queries * A.g * A.nk * (wide ? 1.9e-6 : 0.8e-6));
  const double gather = queries * ((A.g + 3) / 4) * (wide ? 0.0046 * keys / 64 + 0.012 : 0.0014 * keys / 64 + 0.003);
  return tiles < gather;
}

}  // namespace nsa

using namespace nsa;

static int dense_args_f32(const nsa_dense_desc* d, const float* mem_k, const float* mem_v, int32_t q_offset, F32Args& A) {
  const int rc = f32_common(d->batch, d->kv_heads, d->group, d->seq, q_offset, d->dim_head, d->scale, d->q_stride, d->k_stride, d->v_stride, A);
  if (rc) return rc;
  if (d->num_keys < 0 || d->num_mem < 0 || d->num_mem > 64) return NSA_E_ARG;
  A.nk = d->num_keys; A.mem = d->num_mem; A.mode = d->mode; A.causal = d->causal ? 1 : 0;
  A.wb = A.wf = 0; A.st = 1;
  A.memk = mem_k; A.memv = mem_v;
  if (d->mode == 0) {
    if (d->window < 0 || d->num_mem != 0) return NSA_E_ARG;
    A.wb = d->window; A.wf = A.causal ? 0 : d->window;
  } else if (d->mode == 1) {
    if (d->stride <= 0) return NSA_E_ARG;
    if (A.causal && A.mem == 0) return NSA_E_ARG;
    A.st = d->stride;
  } else {
    return NSA_E_ARG;
  }
  return 0;
}

static int dense_fwd_f32(const nsa_dense_desc* d, const float* q, const float* k, const float* v, const float* mem_k, const float* mem_v, float* out,
                         float* lse, int32_t q_offset, void* stream) {
  if (!d || !q || !k || !v || !out) return NSA_E_ARG;
  F32Args A{};
  if (const int rc = dense_args_f32(d, mem_k, mem_v, q_offset, A)) return rc;
  if (!f32_tiles_fit(A)) {
    f32_launch_rows<false>(A, q, k, v, nullptr, nullptr, out, lse, (hipStream_t)stream);
  } else {
    f32_launch_tiles<false>(A, q, k, v, nullptr, nullptr, out, lse, (hipStream_t)stream);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

extern "C" int nsa_dense_fwd_f32(const nsa_dense_desc* d, const float* q, const float* k, const float* v, float* out, float* lse,
                                 int32_t q_offset, void* stream) {
  return dense_fwd_f32(d, q, k, v, nullptr, nullptr, out, lse, q_offset, stream);
}

extern "C" int nsa_compress_fwd_f32(const nsa_dense_desc* d, const float* q, const float* k, const float* v, const float* mem_k, const float* mem_v,
                                    float* out, float* lse, int32_t q_offset, void* stream) {
  if (!d || d->mode != 1 || d->num_mem <= 0 || !mem_k || !mem_v || ((reinterpret_cast<uintptr_t>(mem_k) | reinterpret_cast<uintptr_t>(mem_v)) & 15))
    return NSA_E_ARG;
  return dense_fwd_f32(d, q, k, v, mem_k, mem_v, out, lse, q_offset, stream);
}

extern "C" int nsa_selftest_f32_tiles(int32_t pairs, int32_t tiles, int32_t two_to_a_cu, int32_t* out) {
  if (!out || pairs <= 0 || tiles <= 0) return NSA_E_ARG;
  for (int id = 0; id < pairs * tiles; ++id) {
    const TilePlace at = f32_tile_place(id, pairs * tiles, pairs, two_to_a_cu != 0);
    out[id] = at.pair * tiles + at.tile;
  }
  return 0;
}

extern "C" int nsa_compress_window_fwd_f32(const nsa_dense_desc* dc, const float* q, const float* ck, const float* cv, const float* mem_k, const float* mem_v,
                                           float* out_c, const nsa_dense_desc* dw, const float* rq, const float* k, const float* v, float* out_w,
                                           void* stream) {
  if (!dc || !dw || !q || !ck || !cv || !mem_k || !mem_v || !out_c || !rq || !k || !v || !out_w) return NSA_E_ARG;
  if (dc->mode != 1 || dc->num_mem <= 0 || dw->mode != 0 || ((reinterpret_cast<uintptr_t>(mem_k) | reinterpret_cast<uintptr_t>(mem_v)) & 15)) return NSA_E_ARG;
  RowsCall X{}, Y{};
  if (const int rc = dense_args_f32(dc, mem_k, mem_v, 0, X.A)) return rc;
  if (const int rc = dense_args_f32(dw, nullptr, nullptr, 0, Y.A)) return rc;
  if (X.A.n != Y.A.n || X.A.b != Y.A.b || X.A.hk != Y.A.hk || X.A.g != Y.A.g || X.A.d != Y.A.d) return NSA_E_ARG;
  if (f32_tiles_fit(X.A)) {
    if (const int rc = dense_fwd_f32(dc, q, ck, cv, mem_k, mem_v, out_c, nullptr, 0, stream)) return rc;
    return dense_fwd_f32(dw, rq, k, v, nullptr, nullptr, out_w, nullptr, 0, stream);
  }
  X.q = q; X.k = ck; X.v = cv; X.out = out_c;
  Y.q = rq; Y.k = k; Y.v = v; Y.out = out_w;
  const bool shared = (long)X.A.n * X.A.b * X.A.hk < 1024;            // (as f32_launch_rows)
  const dim3 grid(shared ? X.A.n : (X.A.n + 3) / 4, X.A.b * X.A.hk, 2);
  hipStream_t st = (hipStream_t)stream;
  if (X.A.d <= 64) {
    if (shared) hipLaunchKernelGGL((f32_rows_pair_kernel<1, 4>), grid, dim3(256), 0, st, X, Y);
    else hipLaunchKernelGGL((f32_rows_pair_kernel<1, 1>), grid, dim3(256), 0, st, X, Y);
  } else {
    if (shared) hipLaunchKernelGGL((f32_rows_pair_kernel<2, 4>), grid, dim3(256), 0, st, X, Y);
    else hipLaunchKernelGGL((f32_rows_pair_kernel<2, 1>), grid, dim3(256), 0, st, X, Y);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

extern "C" int nsa_select_fwd_f32(const nsa_select_desc* d, const float* q, const float* k, const float* v, const void* idx,
                                  const uint8_t* fmask, float* out, float* lse, int32_t num_keys, int32_t q_offset, void* stream) {
  if (!d || !q || !k || !v || !out) return NSA_E_ARG;
  F32Args A{};
  const int rc = f32_common(d->batch, d->kv_heads, d->group, d->seq, q_offset, d->dim_head, d->scale, d->q_stride, d->k_stride, d->v_stride, A);
  if (rc) return rc;
  if (d->num_sel < 0 || d->block <= 0 || (d->num_sel > 0 && (!idx || !fmask))) return NSA_E_ARG;
  if (num_keys <= 0 || (d->causal && d->seq + q_offset > num_keys)) return NSA_E_ARG;      // a query's own position must have a key row
  A.nk = num_keys; A.S = d->num_sel; A.B = d->block; A.W = (num_keys + d->block - 1) / d->block; A.causal = d->causal ? 1 : 0;
  A.idx64 = d->idx_is_int64 ? 1 : 0;
  A.uniform = !A.causal && A.S > 0 && q_offset == 0 && num_keys == d->seq;
  if (f32_masked_tiles(A)) f32_launch_tiles<true>(A, q, k, v, idx, fmask, out, lse, (hipStream_t)stream);
  else f32_launch_rows<true>(A, q, k, v, idx, fmask, out, lse, (hipStream_t)stream);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}
