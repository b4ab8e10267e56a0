// fp32 matrix products for the projections of fp32 modules, y = x w^T (+ bias, ReLU), on the bf16 matrix instructions with
// operands split in three (nsa_split.hpp, also for what the sums' error is).  Bound by the matrix instructions, 0.5 of their rate at
// 8192 x 4096 -> 6144 (2460 us, 1.34 PFLOP/s of bf16 products; the library's fp32 kernel 2736 us).
//
// A work-group of four waves (2 x 2) makes a 128 x 128 tile of y, sixteen of the contraction index at a time: while the products of one
// step are made from one set of LDS planes, the next step passes from registers through the split into the other, piece by piece
// between the products, and the one after the next is on its way from memory.  Two work-groups share a CU.
#include <initializer_list>
#include <type_traits>
#include "nsa_split.hpp"
#include "../../include/nsa_hip.h"

namespace nsa {

struct GemmPart { const float *x, *w, *bias; float* y; };
struct GemmArgs {
  GemmPart part[2];              // products of the same sizes, one after the other in the grid
  int m, n, k, relu, tiles_n, tiles;      // tiles: of both
  long ldx;
};

constexpr int kGemmBK = 16, kGemmTile = 128;
constexpr int kGemmPitch = 24;   // elements of an LDS row: 48 bytes, the 16-byte reads of 16 rows touch every bank once
constexpr int kGemmPlane = kGemmTile * kGemmPitch;

// One operand's 16 columns of 128 rows on their way: 4 threads to a row, a thread has two pieces of 16 bytes.
struct GemmOperand {
  const float* base;               // wave-uniform: the tile's first row at contraction index 0
  unsigned off[2];                 // this thread's pieces from there (rows past the last re-read it: their results are not stored)
  int at[2], piece;

  __device__ __forceinline__ void init(const float* p, long ld, int row0, int rows, int tid) {
    base = p + (long)row0 * ld;
    piece = tid % 4;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = u * 64 + tid / 4;
      off[u] = (unsigned)min(r, rows - 1 - row0) * (unsigned)ld + 4 * piece;
      at[u] = r * kGemmPitch + 4 * piece;
    }
  }
  // indices k .. k + 15 (TAIL: those from the end on are zeros)
  template <bool TAIL>
  __device__ __forceinline__ floatx4 load(int u, int k, int end) const {
    if (!TAIL) return *reinterpret_cast<const floatx4*>(base + k + off[u]);
    const int kk = k + 4 * piece;
    floatx4 x = *reinterpret_cast<const floatx4*>(base + (min(kk, end - 4) - 4 * piece) + (long)off[u]);      // (`end` is a multiple of 4)
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = kk < end ? x[e] : 0.f;
    return x;
  }
  __device__ __forceinline__ void put(int u, floatx4 x, __bf16* planes) const {
    const Split3 s = split4(x);
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<bf16x4*>(planes + at[u] + pl * kGemmPlane) = s.part[pl];
  }
};

template <bool TAIL>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(const GemmArgs G) {
  __shared__ __align__(16) __bf16 a_s[2][3 * kGemmPlane], b_s[2][3 * kGemmPlane];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n_ = lane & 31, h = lane >> 5;
  // Work-group ids go round-robin over the 8 XCDs: each gets one run of tiles, row by row, so that its L2 holds a few rows of x
  // tiles and w
  const int id = blockIdx.x, per = G.tiles / 8, rest = G.tiles % 8, x = id & 7, nth = id >> 3;
  int tile = x * per + min(x, rest) + nth;
  const int half = G.part[1].x != nullptr ? G.tiles / 2 : G.tiles;
  const GemmPart P = tile < half ? G.part[0] : G.part[1];
  tile = tile < half ? tile : tile - half;
  const int row0 = (tile / G.tiles_n) * kGemmTile, col0 = (tile % G.tiles_n) * kGemmTile;
  const int steps = (G.k + kGemmBK - 1) / kGemmBK;

  GemmOperand A, B;
  A.init(P.x, G.ldx, row0, G.m, tid);
  B.init(P.w, G.k, col0, G.n, tid);
  // (steps past the last one fetch the last one again)
  auto index = [&](int t) { return kGemmBK * min(t, steps - 1); };
  floatx4 xa[2][2], xb[2][2];
  auto fetch = [&](int t, floatx4 (&ra)[2], floatx4 (&rb)[2]) {
    const int k = index(t);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      ra[u] = A.load<TAIL>(u, k, G.k);
      rb[u] = B.load<TAIL>(u, k, G.k);
    }
  };
  fetch(0, xa[0], xb[0]);
  fetch(1, xa[1], xb[1]);

  floatx16 lead[2][2], small[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) { lead[i][j] = zero_acc(); small[i][j] = zero_acc(); }
#pragma unroll
  for (int u = 0; u < 2; ++u) { A.put(u, xa[0][u], a_s[0]); B.put(u, xb[0][u], b_s[0]); }
  fetch(2, xa[0], xb[0]);
  __syncthreads();

  const int a_at = ((wave >> 1) * 64 + n_) * kGemmPitch + 8 * h, b_at = ((wave & 1) * 64 + n_) * kGemmPitch + 8 * h;
  bf16x8 fa[3][2], fb[3][2];
  auto read = [&](int pl, int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      fa[pl][i] = *reinterpret_cast<const bf16x8*>(a_s[buf] + a_at + pl * kGemmPlane + 32 * i * kGemmPitch);
      fb[pl][i] = *reinterpret_cast<const bf16x8*>(b_s[buf] + b_at + pl * kGemmPlane + 32 * i * kGemmPitch);
    }
  };
  auto products = [&](int p, int q, floatx16 (&acc)[2][2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(fa[p][i], fb[q][j], acc[i][j]);
  };
  read(0, 0);
  // Step t: products from planes BUF, which hold it (the leading parts' operands are in registers already).  The last step splits a
  // copy of itself that nobody reads.
  auto step = [&](auto buf, int t) {
    constexpr int BUF = decltype(buf)::value;
    floatx4 (&ra)[2] = xa[BUF ^ 1];
    floatx4 (&rb)[2] = xb[BUF ^ 1];
    const int knext = index(t + 3);
    read(2, BUF);
    read(1, BUF);
    products(0, 0, lead);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      A.put(u, ra[u], a_s[BUF ^ 1]);
      ra[u] = A.load<TAIL>(u, knext, G.k);
    }
    products(0, 2, small);
    products(2, 0, small);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      B.put(u, rb[u], b_s[BUF ^ 1]);
      rb[u] = B.load<TAIL>(u, knext, G.k);
    }
    products(0, 1, small);
    products(1, 0, small);
#pragma unroll
    for (int i = 0; i < 20; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // an MFMA,
      __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);       // six vector instructions
    }
    __syncthreads();
    read(0, BUF ^ 1);
    products(1, 1, small);
    products(1, 2, small);
    products(2, 1, small);
  };
  int t = 0;
  for (; t + 1 < steps; t += 2) {
    step(std::integral_constant<int, 0>{}, t);
    step(std::integral_constant<int, 1>{}, t + 1);
  }
  if (t < steps) step(std::integral_constant<int, 0>{}, t);

#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = col0 + (wave & 1) * 64 + 32 * j + n_;
    if (col >= G.n) continue;
    const float add = P.bias != nullptr ? P.bias[col] : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = row0 + (wave >> 1) * 64 + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
        if (row >= G.m) continue;
        float y = split_sum(lead[i][j][e], small[i][j][e]) + add;
        if (G.relu) y = y < 0.f ? 0.f : y;               // (a NaN stays)
        P.y[(long)row * G.n + col] = y;
      }
  }
}

}  // namespace nsa

using namespace nsa;

extern "C" int nsa_gemm_f32(int32_t m, int32_t k, int32_t n, const float* x, int64_t ldx, const float* w, const float* bias, int32_t relu, float* y,
                            const float* x2, const float* w2, const float* bias2, float* y2, void* stream) {
  if (!x || !w || !y || m <= 0 || n <= 0 || k < 4 || (k & 3) || ldx < k || (ldx & 3) || ldx >> 24 || k >> 24) return NSA_E_ARG;
  if ((x2 != nullptr) != (w2 != nullptr) || (x2 != nullptr) != (y2 != nullptr) || (!x2 && bias2)) return NSA_E_ARG;
  for (const float* p : {x, w, x2, w2})
    if (reinterpret_cast<uintptr_t>(p) & 15) return NSA_E_ARG;
  GemmArgs G{};
  G.part[0] = GemmPart{x, w, bias, y};
  G.part[1] = GemmPart{x2, w2, bias2, y2};
  G.m = m; G.n = n; G.k = k; G.ldx = ldx; G.relu = relu;
  const long tm = ((long)m + kGemmTile - 1) / kGemmTile, tn = ((long)n + kGemmTile - 1) / kGemmTile;
  if (tm * tn > 0x3fffffffL) return NSA_E_UNSUPPORTED;
  G.tiles_n = (int)tn; G.tiles = (int)(tm * tn) * (x2 ? 2 : 1);
  if (k % kGemmBK) hipLaunchKernelGGL(gemm_f32_kernel<true>, dim3(G.tiles), dim3(256), 0, (hipStream_t)stream, G);
  else hipLaunchKernelGGL(gemm_f32_kernel<false>, dim3(G.tiles), dim3(256), 0, (hipStream_t)stream, G);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}
