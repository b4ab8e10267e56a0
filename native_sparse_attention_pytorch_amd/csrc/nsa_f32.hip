// fp32 forward kernels: the attention branches evaluated entirely in fp32 (products, softmax,
// accumulation), for fp32 modules, whose outputs must agree with the reference's fp32 torch path
// to its own test tolerance (1e-5, tests/test_sparse_attn.py:86).  The bf16 MFMA kernels cannot give
// that.  They follow the same contracts as nsa_select_fwd (NSA.py:741-819) and nsa_dense_fwd
// (NSA.py:153-184, 632-639, 841-850): any head dimension <= 128 that is a multiple of 4, any group
// size, any block size.
//
// Two kernels, both on the fp32 matrix instructions (256 FLOP per cycle and CU, twice what scalar FMAs reach):
//  * f32_tile_kernel  - interval masks (band, strided prefix): 32 rows (query, head) per wave against
//    32-key tiles shared by the work-group, v_mfma_f32_32x32x2;
//  * f32_rows_kernel  - one query of one kv head per wave (or per work-group) against 64-key tiles gathered
//    from anywhere, v_mfma_f32_4x4x1 with 16 blocks = 64 keys x 4 heads: block selection, and interval
//    masks with few queries (decode steps).
#include <type_traits>
#include "nsa_common.hpp"
#include "../../include/nsa_hip.h"

namespace nsa {

constexpr int kF32MaxD = 128;

struct F32Args {
  int b, hk, g, n, nk, d;          // n: number of queries (rows of q / out); nk: key rows after the memory slots
  int qoff;                       // query row i sits at sequence position i + qoff
  float scale;
  long sq[3], sk[3], sv[3];
  // dense
  int mode, causal, wb, wf, st, mem;
  const float *memk, *memv;       // the memory rows [hk, mem, d] when they are not the first rows of k / v, else null
  // selection
  int S, B, W, idx64, uniform;
};

__device__ __forceinline__ floatx16 mfma32x2(float a, float b, floatx16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

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
template <int DT, bool SELECT, int WPQ>
__global__ __launch_bounds__(256, 2) void f32_rows_kernel(const F32Args A, const float* __restrict__ q, const float* __restrict__ k,
                                                          const float* __restrict__ v, const void* __restrict__ idx,
                                                          const uint8_t* __restrict__ fmask, float* __restrict__ out, float* __restrict__ lse) {
  __shared__ float pieces[4 * kRowsPiece];
  __shared__ int blocks_s[4][64], rows_s[4][64];
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

// ------------------------------------------------------------------------------------------ tile
//
// Interval masks with many queries: a wave holds 32 rows (row r of a kv head = query r / G, head r % G, so any group size
// fits), a work-group 128; tiles of 32 keys of K and V are shared through LDS, double-buffered, one barrier per tile.
//   S^T = K Q^T: A = K (lane = key, half h: features 8 t + 4 h + j in step j of group t), B = Q in the same order;
//   O^T = V^T P^T: step i takes the keys that register i of S^T holds, 8 (i / 4) + 4 h + i % 4, so P goes in as it is.
// 64 MFMAs of 64 cycles per tile at d = 64: bound by the fp32 matrix rate (154 TFLOP/s by a large library GEMM).  Window 512, 4
// heads x 4 kv heads, d = 64, 4096 queries: 0.104 ms (2.28 ms one query per wave in scalar FMAs), 8.6 GFLOP in 32-key tiles.
// (Looking every value over for infinities and NaN on its way into LDS costs 0 to 1.5 %: window 512, 4 heads x 8 kv heads, d = 128, 4096
// queries 366 -> 371 us.)

template <int D>
__global__ __launch_bounds__(256, 2) void f32_tile_kernel(const F32Args A, const float* __restrict__ q, const float* __restrict__ k,
                                                          const float* __restrict__ v, float* __restrict__ out, float* __restrict__ lse) {
  constexpr int VS = D + 8;                              // V row stride: the halves' rows (4 apart) lie 32 banks apart
  constexpr int LD = D / 32;                             // 16-byte loads per thread and tile of K (and of V)
  __shared__ float k_s[2][32 * D];                       // chunk c of row r at c ^ (r % 16)
  __shared__ float v_s[2][32 * VS];                      // (zeros for values that are not finite)
  __shared__ int odd_s;                                  // there was such a value
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n_ = lane & 31, h = lane >> 5;
  const int bh = blockIdx.y, b = bh / A.hk, hk = bh % A.hk;
  const float* kb = k + b * A.sk[0] + hk * A.sk[1];
  const float* vb = v + b * A.sv[0] + hk * A.sv[1];
  const long all_rows = (long)A.n * A.g;
  const long row0 = (long)(gridDim.x - 1 - blockIdx.x) * 128;              // longest key lists first (causal prefixes)
  const long row = row0 + wave * 32 + n_;
  const long rowc = row < all_rows ? row : all_rows - 1;
  const int qi = (int)(rowc / A.g), g = (int)(rowc - (long)qi * A.g);
  int lo, hi;
  f32_interval(A, qi + A.qoff, lo, hi);
  // ranges of the wave's and of the work-group's rows (both ends grow with the query)
  const int wq0 = (int)(min(row0 + wave * 32, all_rows - 1) / A.g), wq1 = (int)(min(row0 + wave * 32 + 31, all_rows - 1) / A.g);
  const int gq0 = (int)(row0 / A.g), gq1 = (int)(min(row0 + 127, all_rows - 1) / A.g);
  int w_lo0, w_hi1, g_lo, g_hi, dummy;
  f32_interval(A, wq0 + A.qoff, w_lo0, dummy);
  f32_interval(A, wq1 + A.qoff, dummy, w_hi1);
  f32_interval(A, gq0 + A.qoff, g_lo, dummy);
  f32_interval(A, gq1 + A.qoff, dummy, g_hi);
  if (A.mode == 1) { w_hi1 = max(w_hi1, A.mem - 1); g_hi = max(g_hi, A.mem - 1); }
  hi = A.mode == 1 ? max(hi, A.mem - 1) : hi;
  // a key is visible if key - lo, as an unsigned number, is at most `seen`: one comparison, and no branch per element
  const unsigned seen = hi < lo ? 0u : (unsigned)(hi - lo);
  if (hi < lo) lo = 0x7fffffff;

  float qr[D / 8][4];
  {
    const float* qp = q + b * A.sq[0] + (long)(hk * A.g + g) * A.sq[1] + (long)qi * A.sq[2];
#pragma unroll
    for (int t = 0; t < D / 8; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) qr[t][j] = qp[min(8 * t + 4 * h + j, A.d - 1)];      // (features past the head dimension meet zero keys)
  }
  floatx16 o[D / 32];
#pragma unroll
  for (int ft = 0; ft < D / 32; ++ft) o[ft] = zero_acc();
  float m = -INFINITY, l = 0.f;

  const int own_mem = A.memk != nullptr ? A.mem : 0;
  floatx4 kx[LD], vx[LD];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int u = 0; u < LD; ++u) {
      const int e = u * 256 + tid, r = e / (D / 4), c = e % (D / 4);
      const int kr = t0 + r;
      floatx4 z = {0.f, 0.f, 0.f, 0.f};
      kx[u] = z;
      vx[u] = z;
      if (kr <= g_hi && 4 * c < A.d) {
        const bool own = kr < own_mem;
        kx[u] = *reinterpret_cast<const floatx4*>((own ? A.memk + ((long)hk * A.mem + kr) * A.d : kb + (long)(kr - own_mem) * A.sk[2]) + 4 * c);
        vx[u] = *reinterpret_cast<const floatx4*>((own ? A.memv + ((long)hk * A.mem + kr) * A.d : vb + (long)(kr - own_mem) * A.sv[2]) + 4 * c);
      }
    }
  };
  const int t_first = g_lo & ~31;
  fetch(t_first);
  if (tid == 0) odd_s = 0;
  __syncthreads();
  bool odd = false;
  int buf = 0;
  for (int t0 = t_first; t0 <= g_hi; t0 += 32, buf ^= 1) {
#pragma unroll
    for (int u = 0; u < LD; ++u) {
      const int e = u * 256 + tid, r = e / (D / 4), c = e % (D / 4);
      *reinterpret_cast<floatx4*>(&k_s[buf][r * D + 4 * (c ^ (r & 15))]) = kx[u];
      floatx4 x;
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        const bool finite = fabsf(vx[u][e2]) < INFINITY;
        odd |= !finite;
        x[e2] = finite ? vx[u][e2] : 0.f;
      }
      *reinterpret_cast<floatx4*>(&v_s[buf][r * VS + 4 * c]) = x;
    }
    __syncthreads();          // (the other buffer was read before this barrier by every wave: it may be written in the next round)
    if (t0 + 32 <= g_hi) fetch(t0 + 32);
    if (t0 > w_hi1 || t0 + 31 < w_lo0) continue;         // wave-uniform: nothing of this tile is visible to the wave
    floatx16 s = zero_acc();
    // (the K operands of 8 feature groups are read ahead of the first product that needs them: at one or two waves per SIMD an
    // LDS round trip in front of every fourth MFMA is not hidden by other waves)
#pragma unroll
    for (int t8 = 0; t8 < D / 8; t8 += 8) {
      floatx4 kk[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) kk[t] = *reinterpret_cast<const floatx4*>(&k_s[buf][n_ * D + 4 * ((2 * (t8 + t) + h) ^ (n_ & 15))]);
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) s = mfma32x2(kk[t][j], qr[t8 + t][j], s);
    }
    float sv[16], tmax = -INFINITY;
    const int from_lo = t0 + 4 * h - lo;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      sv[i] = (unsigned)(from_lo + 8 * (i / 4) + (i % 4)) <= seen ? s[i] * A.scale : -INFINITY;
      tmax = fmaxf(tmax, sv[i]);
    }
    tmax = halves_max(tmax);
    const float mn = fmaxf(m, tmax), mref = mn == -INFINITY ? 0.f : mn;
    const float alpha = expf(m - mref);                  // m = -inf: 0
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) { sv[i] = expf(sv[i] - mref); ps += sv[i]; }
    l = l * alpha + ps;                                  // this half's keys
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int ft = 0; ft < D / 32; ++ft)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[ft][i] *= alpha;
    }
#pragma unroll
    for (int i8 = 0; i8 < 16; i8 += 8) {
      float vv[8][D / 32];
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int ft = 0; ft < D / 32; ++ft) vv[i][ft] = v_s[buf][(8 * ((i8 + i) / 4) + 4 * h + (i % 4)) * VS + 32 * ft + n_];
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int ft = 0; ft < D / 32; ++ft) o[ft] = mfma32x2(vv[i][ft], sv[i8 + i], o[ft]);
    }
  }
  // A value that is not finite is left out of the products, where a weight of zero times it would be NaN in every row of its tile,
  // and added here to the rows that see its key.
  if (odd) odd_s = 1;
  __syncthreads();
  if (odd_s) {
#pragma unroll 1
    for (int kr = g_lo; kr <= g_hi; ++kr) {
      const float* vr = kr < own_mem ? A.memv + ((long)hk * A.mem + kr) * A.d : vb + (long)(kr - own_mem) * A.sv[2];
      const bool visible = (unsigned)(kr - lo) <= seen;
#pragma unroll
      for (int ft = 0; ft < D / 32; ++ft)
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
  for (int ft = 0; ft < D / 32; ++ft)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int f0 = 32 * ft + 8 * u + 4 * h;
      if (f0 < A.d)
        *reinterpret_cast<floatx4*>(op + f0) = floatx4{o[ft][4 * u] * inv, o[ft][4 * u + 1] * inv, o[ft][4 * u + 2] * inv, o[ft][4 * u + 3] * inv};
    }
  if (lse != nullptr && h == 0) lse[orow] = l > 0.f ? m + logf(l) : -INFINITY;
}

static int f32_common(int batch, int kv_heads, int group, int seq, int q_offset, int dim_head, float scale, const int64_t* qs, const int64_t* ks,
                      const int64_t* vs, F32Args& A) {
  if (batch <= 0 || kv_heads <= 0 || group <= 0 || seq <= 0 || q_offset < 0) return NSA_E_ARG;
  A.qoff = q_offset;
  if (dim_head <= 0 || dim_head > kF32MaxD || (dim_head & 3)) return NSA_E_UNSUPPORTED;
  if ((long)batch * kv_heads > 65535) return NSA_E_UNSUPPORTED;
  A.b = batch; A.hk = kv_heads; A.g = group; A.n = seq; A.d = dim_head; A.scale = scale;
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

}  // namespace nsa

using namespace nsa;

static int dense_fwd_f32(const nsa_dense_desc* d, const float* q, const float* k, const float* v, const float* mem_k, const float* mem_v, float* out,
                         float* lse, int32_t q_offset, void* stream) {
  if (!d || !q || !k || !v || !out) return NSA_E_ARG;
  F32Args A{};
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
  // A wave of the tile kernel takes 32 rows through all their keys: below ~4096 queries too few waves with too long a walk.
  // Window 512, d = 64, 4 heads: 2048 queries 65 us in tiles, 41 us row by row; 4096 queries 65 against 82 us.
  if ((long)A.n * A.b * A.hk < 4096) {
    f32_launch_rows<false>(A, q, k, v, nullptr, nullptr, out, lse, (hipStream_t)stream);
  } else {
    const dim3 grid((unsigned)(((long)A.n * A.g + 127) / 128), A.b * A.hk);
    if (A.d <= 64) hipLaunchKernelGGL(f32_tile_kernel<64>, grid, dim3(256), 0, (hipStream_t)stream, A, q, k, v, out, lse);
    else hipLaunchKernelGGL(f32_tile_kernel<128>, grid, dim3(256), 0, (hipStream_t)stream, A, q, k, v, out, lse);
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
  f32_launch_rows<true>(A, q, k, v, idx, fmask, out, lse, (hipStream_t)stream);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}
