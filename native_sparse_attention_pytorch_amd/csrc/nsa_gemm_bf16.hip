// bf16 matrix products of the trained projections: y = x w^T with its epilogue, the input's gradient dy w, and the weight's gradient dy^T x
// with the bias's beside it.
//
// A work-group of four waves (2 x 2) makes a TM x 128 tile of the result, 64 of the contraction index at a time: both operands' tiles are
// copied straight into swizzled LDS (TileDma) one step ahead, between the matrix instructions of the step in use.  An operand whose rows
// run along the contraction (x and w of y) is read row by row; one whose rows are the contraction index (w of dx, both of dw) through
// the transposing LDS reads, so no operand is laid out anew in memory.  Two work-groups share a CU (64 KB of LDS each).
#include <algorithm>
#include "nsa_common.hpp"
#include "../../include/nsa_hip.h"

namespace nsa {

struct BGemmPart {
  const __bf16 *a, *b, *bias, *act, *residual;      // act: what the backward of the activation reads
  __bf16 *y, *pre;                                  // pre: the value before a GELU
  float *part, *bpart;                              // weight gradient: slices [splits][m][n] and [splits][m]
};
struct BGemmArgs {
  BGemmPart part[2];                                // products of the same sizes, one after the other in the grid
  int m, n, k, epi, tiles_n, tiles, splits, slice, total;      // tiles: of one slice; total: of all
  long lda, ldb;
};

constexpr int kBK64 = 64, kBN = 128;

// As lds_transposed_operand_swz, with the rows in the order of a row operand (8 h + e)
template <int D>
__device__ __forceinline__ bf16x8 lds_transposed_rows(const __bf16* X, int row0, int col0, int lane) {
  const int ll = lane & 15, e = ll >> 2, qq = ll & 3, mh = (lane >> 4) & 1, h = lane >> 5;
  typedef shortx4 __attribute__((address_space(3))) * lds_ptr;
  const int chunk = (col0 >> 3) + 2 * mh + (qq >> 1), at = 4 * (qq & 1);
  const shortx4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(X + lds_swz_off<D>(row0 + 8 * h + e, chunk) + at));
  const shortx4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(X + lds_swz_off<D>(row0 + 8 * h + 4 + e, chunk) + at));
  typedef __attribute__((__vector_size__(8 * sizeof(short)))) short shortx8;
  shortx8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) { r[i] = a[i]; r[4 + i] = b[i]; }
  return __builtin_bit_cast(bf16x8, r);
}

// erfc(|x| / sqrt 2) / 2 by Abramowitz and Stegun's 7.1.26 (an exponential that the slope needs as well and five multiply-adds; the
// library's erff is two branches of twice that, which cost 16 of 44 us at 8192 x 512 -> 2048).  Over |x| < 12 against float64, GELU and
// slope are off by 3.3e-7 and 2.6e-7 at most (torch's fp32 GELU: 1.1e-6, 2.6e-7): 1 + erf does not cancel for negative x here.
struct GaussTail { float q, e; };
__device__ __forceinline__ GaussTail gauss_tail(float x) {
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.3275911f * 0.70710678118654752f, fabsf(x), 1.0f));
  const float e = fast_exp2(-0.5f * kLog2e * x * x);
  float p = __builtin_fmaf(1.061405429f, t, -1.453152027f);
  p = __builtin_fmaf(p, t, 1.421413741f);
  p = __builtin_fmaf(p, t, -0.284496736f);
  p = __builtin_fmaf(p, t, 0.254829592f);
  return GaussTail{0.5f * p * t * e, e};
}
__device__ __forceinline__ float gelu(float x) {
  const float q = gauss_tail(x).q;
  return x * (x > 0.f ? 1.0f - q : q);
}
__device__ __forceinline__ float gelu_slope(float x) {
  const GaussTail g = gauss_tail(x);
  return (x > 0.f ? 1.0f - g.q : g.q) + x * (0.39894228040143268f * g.e);
}

// One operand: R result rows (or columns) by 64 of the contraction index a step
template <bool TRANS, int R>
struct BOperand {
  static constexpr int D = TRANS ? R : 64, TILES = TRANS ? 1 : R / 64, ROUNDS = TILES * TileDma<D, 256>::ROUNDS;
  TileDma<D, 256> dma;
  const __bf16* base;
  long ld;
  int first, limit, kend;
  __device__ __forceinline__ void init(const __bf16* p, long stride, int row0, int rows, int k_end, int tid, const __bf16* lds) {
    dma.init(tid, stride, lds);
    ld = stride; first = row0; limit = rows; kend = k_end;
    base = TRANS ? p + row0 : p;
  }
  // all of the tile at contraction index k exists (in the direction of its rows)
  __device__ __forceinline__ bool whole(int k) const { return TRANS ? k + kBK64 <= kend : first + R <= limit; }
  __device__ __forceinline__ void issue(int k, unsigned off) const {
    if (TRANS) {
      dma.issue(base, k, kend, off);
    } else {
#pragma unroll
      for (int t = 0; t < TILES; ++t) dma.issue(base + k, first + 64 * t, limit, off + t * 64 * 64 * 2);
    }
  }
  __device__ __forceinline__ void round(int k, unsigned off, int r) const {
    if (TRANS) {
      dma.round_full(base + (long)k * ld, off, r);
    } else {
      constexpr int RN = TileDma<D, 256>::ROUNDS;
      dma.round_full(base + k + (long)(first + 64 * (r / RN)) * ld, off + (r / RN) * 64 * 64 * 2, r % RN);
    }
  }
  // the operand of rows (columns) 32 f .. 32 f + 31, indices 16 ks .. 16 ks + 15 of the step
  __device__ __forceinline__ static bf16x8 read(const __bf16* s, int f, int ks, int lane) {
    if (TRANS) return lds_transposed_rows<D>(s, 16 * ks, 32 * f, lane);
    return lds_row_operand_swz<64>(s + 32 * f * 64, ks, lane);
  }
};

// FORM 0: y[m, n] = a[m, k] b[n, k]^T; 1: a[m, k] b[k, n]; 2: a[k, m]^T b[k, n], in slices of the contraction index
template <int FORM, int TM>
__global__ __launch_bounds__(256, 2) void gemm_bf16_kernel(const BGemmArgs G) {
  constexpr int MI = TM / 64, ATILE = TM * kBK64, BTILE = kBN * kBK64;
  typedef BOperand<FORM == 2, TM> OpA;
  typedef BOperand<FORM != 0, kBN> OpB;
  __shared__ __align__(1024) __bf16 a_s[2 * ATILE + 2 * BTILE];
  __bf16* b_s = a_s + 2 * ATILE;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n_ = lane & 31, h = lane >> 5, wm = wave >> 1, wn = wave & 1;
  // one run of tiles to each XCD: see gemm_f32_kernel
  const int id = blockIdx.x, per = G.total / 8, rest = G.total % 8, x = id & 7;
  int nth = x * per + min(x, rest) + (id >> 3);
  const BGemmPart P = nth < G.tiles * G.splits ? G.part[0] : G.part[1];
  nth = nth < G.tiles * G.splits ? nth : nth - G.tiles * G.splits;
  const int slice = nth / G.tiles, tile = nth % G.tiles;
  const int row0 = (tile / G.tiles_n) * TM, col0 = (tile % G.tiles_n) * kBN;
  const int kbeg = slice * G.slice, kend = min(G.k, kbeg + G.slice);
  const int steps = (kend - kbeg + kBK64 - 1) / kBK64;

  OpA A;
  OpB B;
  A.init(P.a, G.lda, row0, G.m, kend, tid, a_s);
  B.init(P.b, G.ldb, col0, G.n, kend, tid, b_s);
  floatx16 acc[MI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero_acc();
  float bsum[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) bsum[i] = 0.f;
  const bool sums = FORM == 2 && P.bpart != nullptr && col0 == 0 && wn == 0;      // wave-uniform

  A.issue(kbeg, 0);
  B.issue(kbeg, 0);
  for (int t = 0; t < steps; ++t) {
    const int buf = t & 1, k = kbeg + t * kBK64, kn = k + kBK64;
    wait_all_loads();
    __syncthreads();
    __bf16* as = a_s + buf * ATILE;
    __bf16* bs = b_s + buf * BTILE;
    if (FORM == 2 && kn > kend) {            // the rows past the last one are zeros
      for (int e = tid; e < (kn - kend) * (OpA::D / 8); e += 256) *reinterpret_cast<bf16x8*>(as + (kend - k) * OpA::D + 8 * e) = zero_frag();
      for (int e = tid; e < (kn - kend) * (OpB::D / 8); e += 256) *reinterpret_cast<bf16x8*>(bs + (kend - k) * OpB::D + 8 * e) = zero_frag();
      __syncthreads();
    }
    const bool more = t + 1 < steps, spread = more && A.whole(kn) && B.whole(kn);
    const unsigned aoff = (buf ^ 1) * ATILE * 2, boff = (buf ^ 1) * BTILE * 2;
    if (more && !spread) {
      A.issue(kn, aoff);
      B.issue(kn, boff);
    }
    auto products = [&](auto copying) {
      bf16x8 fa[2][MI], fb[2][2];
      auto read = [&](int ks, int into) {
#pragma unroll
        for (int i = 0; i < MI; ++i) fa[into][i] = OpA::read(as, wm * MI + i, ks, lane);
#pragma unroll
        for (int j = 0; j < 2; ++j) fb[into][j] = OpB::read(bs, wn * 2 + j, ks, lane);
      };
      read(0, 0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        if (ks < 3) read(ks + 1, (ks + 1) & 1);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            acc[i][j] = mfma32(fa[ks & 1][i], fb[ks & 1][j], acc[i][j]);
            constexpr int RA = OpA::ROUNDS, RB = OpB::ROUNDS, EVERY = 8 * MI / (RA + RB);
            const int at = (ks * MI + i) * 2 + j, r = at / EVERY;
            if (decltype(copying)::value && at % EVERY == EVERY - 1 && r < RA + RB) {
              if (r < RA) A.round(kn, aoff, r);
              else B.round(kn, boff, r - RA);
            }
          }
        if (FORM == 2 && sums) {
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) s += (float)fa[ks & 1][i][e];
            bsum[i] += s;
          }
        }
      }
    };
    if (spread) products(std::true_type{});
    else products(std::false_type{});
  }

  if (FORM == 2) {
    float* part = P.part + (size_t)slice * G.m * G.n;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = col0 + wn * 64 + 32 * j + n_;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) part[(size_t)(row0 + wm * (TM / 2) + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3)) * G.n + col] = acc[i][j][e];
    }
    if (sums) {
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const float s = halves_sum(bsum[i]);
        if (h == 0) P.bpart[(size_t)slice * G.m + row0 + wm * (TM / 2) + 32 * i + n_] = s;
      }
    }
    return;
  }
  // the tile through LDS, 32 rows of a wave at a time: 16 bytes of a row to a lane
  __syncthreads();
  constexpr int PITCH = 68;
  float* st = reinterpret_cast<float*>(a_s) + wave * 32 * PITCH;
  const int c8 = 8 * (lane & 7), gcol = col0 + wn * 64 + c8;
  const bool cok = gcol < G.n;
  float add[8];
  {
    const bf16x8 t = cok && P.bias != nullptr ? load8(P.bias + gcol) : zero_frag();
#pragma unroll
    for (int e = 0; e < 8; ++e) add[e] = (float)t[e];
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) st[(8 * (e >> 2) + 4 * h + (e & 3)) * PITCH + 32 * j + n_] = acc[i][j][e];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int r = 8 * p + (lane >> 3), row = row0 + wm * (TM / 2) + 32 * i + r;
      const floatx4 u = *reinterpret_cast<const floatx4*>(st + r * PITCH + c8), w = *reinterpret_cast<const floatx4*>(st + r * PITCH + c8 + 4);
      if (row >= G.m || !cok) continue;
      const long at = (long)row * G.n + gcol;
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (__bf16)((e < 4 ? u[e & 3] : w[e & 3]) + add[e]);
      if (G.epi == NSA_GEMM_RELU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (float)o[e] < 0.f ? (__bf16)0.f : o[e];      // (a NaN stays)
      } else if (G.epi == NSA_GEMM_GELU) {
        if (P.pre != nullptr) *reinterpret_cast<bf16x8*>(P.pre + at) = o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (__bf16)gelu((float)o[e]);
      } else if (G.epi == NSA_GEMM_RELU_BWD) {
        const bf16x8 g = load8(P.act + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (float)g[e] <= 0.f ? (__bf16)0.f : o[e];
      } else if (G.epi == NSA_GEMM_GELU_BWD) {
        const bf16x8 g = load8(P.act + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (__bf16)((e < 4 ? u[e & 3] : w[e & 3]) * gelu_slope((float)g[e]));
      }
      if (P.residual != nullptr) {
        const bf16x8 g = load8(P.residual + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (__bf16)((float)o[e] + (float)g[e]);
      }
      *reinterpret_cast<bf16x8*>(P.y + at) = o;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// dw (and db) from the slices: 8 values a thread
__global__ __launch_bounds__(256) void wgrad_sum_kernel(const BGemmArgs G) {
  const BGemmPart P = blockIdx.y == 0 ? G.part[0] : G.part[1];
  const int splits = G.splits;
  long e = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  const float* src = P.part;
  long size = (long)G.m * G.n;
  __bf16* dst = P.y;
  if (e >= size) {
    e -= size;
    if (P.bpart == nullptr || e >= G.m) return;
    src = P.bpart; size = G.m; dst = P.pre;
  }
  floatx4 x = {0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    x += *reinterpret_cast<const floatx4*>(src + s * size + e);
    y += *reinterpret_cast<const floatx4*>(src + s * size + e + 4);
  }
  bf16x8 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) { o[i] = (__bf16)x[i]; o[4 + i] = (__bf16)y[i]; }
  *reinterpret_cast<bf16x8*>(dst + e) = o;
}

static int wgrad_splits(long rows, int n_out, int n_in) {
  const long tiles = (long)(n_out % 128 ? n_out / 64 : n_out / 128) * (n_in / 128), steps = (rows + 63) / 64;
  long s = std::max<long>(1, std::min<long>(512 / tiles, steps / 4));
  const long per = (steps + s - 1) / s;
  return (int)((steps + per - 1) / per);
}

}  // namespace nsa

using namespace nsa;

static bool aligned16(std::initializer_list<const void*> ps) {
  uintptr_t u = 0;
  for (const void* p : ps) u |= reinterpret_cast<uintptr_t>(p);
  return (u & 15) == 0;
}

extern "C" int nsa_gemm_bf16(int32_t transposed, int32_t m, int32_t n, int32_t k, int32_t epilogue, const void* x, const void* w, const void* bias,
                             const void* act, const void* residual, void* y, void* pre, const void* x2, const void* w2, const void* bias2, const void* act2,
                             void* y2, void* pre2, void* stream) {
  if (!x || !w || !y || m <= 0 || n <= 0 || k <= 0) return NSA_E_ARG;
  if (epilogue < 0 || epilogue > NSA_GEMM_GELU_BWD || (epilogue >= NSA_GEMM_RELU_BWD) != (act != nullptr)) return NSA_E_ARG;
  if (x2 ? !w2 || !y2 || !act2 != !act || !bias2 != !bias || residual : w2 || bias2 || act2 || y2 || pre2) return NSA_E_ARG;
  if (k % 64 || n % 8 || n >> 24 || k >> 24 || (transposed && n % 128)) return NSA_E_UNSUPPORTED;
  if (!aligned16({x, w, bias, act, residual, y, pre, x2, w2, bias2, act2, y2, pre2})) return NSA_E_ARG;
  const int products = x2 ? 2 : 1;
  const long tn = ((long)n + kBN - 1) / kBN;
  long tm = ((long)m + 127) / 128;
  const bool small = tm * tn * products < 512;      // tiles of 64 rows
  if (small) tm = ((long)m + 63) / 64;
  if (tm * tn > 0x3fffffffL) return NSA_E_UNSUPPORTED;
  BGemmArgs G{};
  G.part[0] = BGemmPart{(const __bf16*)x, (const __bf16*)w, (const __bf16*)bias, (const __bf16*)act, (const __bf16*)residual, (__bf16*)y, (__bf16*)pre, nullptr, nullptr};
  G.part[1] = BGemmPart{(const __bf16*)x2, (const __bf16*)w2, (const __bf16*)bias2, (const __bf16*)act2, nullptr, (__bf16*)y2, (__bf16*)pre2, nullptr, nullptr};
  G.m = m; G.n = n; G.k = k; G.epi = epilogue; G.tiles_n = (int)tn; G.tiles = (int)(tm * tn); G.splits = 1; G.slice = k; G.total = G.tiles * products;
  G.lda = k; G.ldb = transposed ? n : k;
  const dim3 grid(G.total), block(256);
  hipStream_t st = (hipStream_t)stream;
  if (small && transposed) hipLaunchKernelGGL((gemm_bf16_kernel<1, 64>), grid, block, 0, st, G);
  else if (small) hipLaunchKernelGGL((gemm_bf16_kernel<0, 64>), grid, block, 0, st, G);
  else if (transposed) hipLaunchKernelGGL((gemm_bf16_kernel<1, 128>), grid, block, 0, st, G);
  else hipLaunchKernelGGL((gemm_bf16_kernel<0, 128>), grid, block, 0, st, G);
  return (int)hipGetLastError();
}

extern "C" int64_t nsa_wgrad_bf16_workspace(int64_t rows, int32_t n_out, int32_t n_in) {
  if (rows <= 0 || rows > 0x7fffffff - 64 || n_out <= 0 || n_in <= 0 || n_out % 64 || n_in % 128 || n_out >> 15 || n_in >> 15) return 0;
  return (int64_t)wgrad_splits(rows, n_out, n_in) * ((int64_t)n_out * n_in + n_out) * 4;
}

extern "C" int nsa_wgrad_bf16(int64_t rows, int32_t n_out, int32_t n_in, const void* dy, int64_t lddy, const void* x, int64_t ldx, void* dw, void* db,
                              const void* dy2, const void* x2, void* dw2, void* db2, float* workspace, void* stream) {
  if (!dy || !x || !dw || !workspace || lddy < n_out || ldx < n_in) return NSA_E_ARG;
  if (dy2 ? !x2 || !dw2 || !db2 != !db : x2 || dw2 || db2) return NSA_E_ARG;
  const int64_t bytes = nsa_wgrad_bf16_workspace(rows, n_out, n_in);
  if (bytes == 0 || lddy % 8 || ldx % 8 || lddy >> 24 || ldx >> 24) return NSA_E_UNSUPPORTED;
  if (!aligned16({dy, x, dw, db, dy2, x2, dw2, db2, workspace})) return NSA_E_ARG;
  const int tm = n_out % 128 ? 64 : 128;
  BGemmArgs G{};
  G.lda = lddy; G.ldb = ldx;
  G.m = n_out; G.n = n_in; G.k = (int)rows;
  G.tiles_n = n_in / kBN; G.tiles = (n_out / tm) * G.tiles_n; G.splits = wgrad_splits(rows, n_out, n_in);
  const long steps = (rows + 63) / 64, mn = (long)n_out * n_in;
  G.slice = (int)((steps + G.splits - 1) / G.splits * 64);
  G.total = G.tiles * G.splits * (dy2 ? 2 : 1);
  float* ws2 = workspace + bytes / 4;
  G.part[0] = BGemmPart{(const __bf16*)dy, (const __bf16*)x, nullptr, nullptr, nullptr, (__bf16*)dw, (__bf16*)db, workspace, db ? workspace + G.splits * mn : nullptr};
  if (dy2)
    G.part[1] = BGemmPart{(const __bf16*)dy2, (const __bf16*)x2, nullptr, nullptr, nullptr, (__bf16*)dw2, (__bf16*)db2, ws2, db2 ? ws2 + G.splits * mn : nullptr};
  hipStream_t st = (hipStream_t)stream;
  if (tm == 64) hipLaunchKernelGGL((gemm_bf16_kernel<2, 64>), dim3(G.total), dim3(256), 0, st, G);
  else hipLaunchKernelGGL((gemm_bf16_kernel<2, 128>), dim3(G.total), dim3(256), 0, st, G);
  if (hipError_t e = hipGetLastError()) return (int)e;
  hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)((mn / 8 + n_out / 8 + 255) / 256), dy2 ? 2 : 1), dim3(256), 0, st, G);
  return (int)hipGetLastError();
}
