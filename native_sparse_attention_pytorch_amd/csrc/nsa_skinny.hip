// Projections of a decode step: y = norm(x) W^T + bias for a handful of rows (one token per sequence, NSA.py:356-364, 545), with
// the RMS norm in front (NSA.py:230) when asked for.
//
// Bound by reading W once: 2 K N bytes.  A work-group of eight waves owns 16 output features and shares the K axis, so 4096
// features are 2048 waves that each request up to 16 KB of W before waiting for the first; the batch is the other side of a
// 16x16x32 MFMA.  While W is on its way the work-group brings x into LDS and norms it there - the norm costs no launch and
// no pass of its own.  The waves' partial sums meet in LDS.
// Measured (weights from HBM, launch included): 4096 -> 6240 with norm, batch 1 14.5 us, batch 8 18.1 us, of which the 51 MB
// of W take 9.8 us at the rate of a large copy (norm kernel + library GEMM: 20.6 / 20.8 us); 4096 -> 4096, batch 1 10.2 us (15.6 us);
// 1024 -> 1584 with norm, batch 16 6.4 us (9.3 us).
#include "nsa_common.hpp"
#include "../../include/nsa_hip.h"

namespace nsa {

constexpr int kSkinnyWaves = 8, kSkinnyThreads = 64 * kSkinnyWaves;
constexpr int kSkinnyAhead = 16;                 // K steps (of 32) whose W operands a wave holds
constexpr size_t kSkinnyLds = 128 << 10;         // of x

// NB: groups of 16 rows
template <int NB>
__global__ __launch_bounds__(kSkinnyThreads, 4) void skinny_linear_kernel(int rows, int K, int N, const __bf16* __restrict__ x, long xs,
                                                                          const __bf16* __restrict__ nw, float eps,
                                                                          const __bf16* __restrict__ w, const __bf16* __restrict__ bias,
                                                                          __bf16* __restrict__ y, long ys) {
  extern __shared__ __align__(16) char lds[];
  __shared__ float ss_s[kSkinnyWaves];
  float (*part_s)[NB][16][17] = reinterpret_cast<float (*)[NB][16][17]>(lds);                                 // [wave]
  __bf16* x_s = reinterpret_cast<__bf16*>(lds + sizeof(float) * kSkinnyWaves * NB * 16 * 17);
  const int RS = K + 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, kq = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int steps = K >> 5, per = (steps + kSkinnyWaves - 1) / kSkinnyWaves;
  const int s0 = wave * per, s1 = min(steps, s0 + per);
  const __bf16* wp = w + (long)min(n0 + r, N - 1) * K + 8 * kq;

  bf16x8 wr[kSkinnyAhead];
  auto fetch = [&](int s) {
#pragma unroll
    for (int u = 0; u < kSkinnyAhead; ++u)
      if (s + u < s1) wr[u] = load8(wp + 32 * (s + u));
  };
  fetch(s0);

  // x: 8, 4, 2 or 1 waves per row, eight features per lane and round
  const int share = rows == 1 ? 8 : rows == 2 ? 4 : rows <= 4 ? 2 : 1, sub = wave % share;
  for (int row0 = 0; row0 < rows; row0 += kSkinnyWaves / share) {            // (every wave takes every round: the barrier)
    const int row = row0 + wave / share;
    __bf16* xw = x_s + row * RS;
    float ss = 0.f;
    if (row < rows) {
#pragma unroll 8
      for (int c = 64 * sub + lane; c < K / 8; c += 64 * share) {
        const bf16x8 t = load8(x + row * xs + 8 * c);
        *reinterpret_cast<bf16x8*>(xw + 8 * c) = t;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)t[e] * (float)t[e];
      }
    }
    if (nw != nullptr) {
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
      if (share > 1) {                                                       // (a single round)
        if (lane == 0) ss_s[wave] = ss;
        __syncthreads();
        ss = 0.f;
        for (int v = 0; v < share; ++v) ss += ss_s[wave - sub + v];
      }
      if (row < rows) {
        const float rs = rsqrtf(ss / (float)K + eps);
#pragma unroll 4
        for (int c = 64 * sub + lane; c < K / 8; c += 64 * share) {          // (the chunks this lane wrote)
          bf16x8 t = *reinterpret_cast<const bf16x8*>(xw + 8 * c);
          const bf16x8 n8 = load8(nw + 8 * c);
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = (__bf16)((float)t[e] * rs * (float)n8[e]);      // rounded as a norm of its own would
          *reinterpret_cast<bf16x8*>(xw + 8 * c) = t;
        }
      }
    }
  }
  __syncthreads();

  floatx4 acc[NB];
  const __bf16* xr[NB];
#pragma unroll
  for (int g = 0; g < NB; ++g) {
    acc[g] = floatx4{0.f, 0.f, 0.f, 0.f};
    xr[g] = x_s + min(16 * g + r, rows - 1) * RS + 8 * kq;                   // (columns past the batch repeat its last row, unused)
  }
  for (int s = s0; s < s1; s += kSkinnyAhead) {
#pragma unroll
    for (int u = 0; u < kSkinnyAhead; ++u)
      if (s + u < s1) {                                                      // wave-uniform
#pragma unroll
        for (int g = 0; g < NB; ++g)
          acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[u], *reinterpret_cast<const bf16x8*>(xr[g] + 32 * (s + u)), acc[g], 0, 0, 0);
      }
    if (s + kSkinnyAhead < s1) fetch(s + kSkinnyAhead);
  }
  // D: feature 4 kq + i, batch row r
#pragma unroll
  for (int g = 0; g < NB; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i) part_s[wave][g][r][4 * kq + i] = acc[g][i];
  __syncthreads();
  for (int e = threadIdx.x; e < NB * 256; e += kSkinnyThreads) {
    const int f = e & 15, br = (e >> 4) & 15, g = e >> 8;
    if (16 * g + br >= rows || n0 + f >= N) continue;
    float t = 0.f;
#pragma unroll
    for (int v = 0; v < kSkinnyWaves; ++v) t += part_s[v][g][br][f];
    if (bias != nullptr) t += (float)bias[n0 + f];
    y[(long)(16 * g + br) * ys + n0 + f] = (__bf16)t;
  }
}

}  // namespace nsa

extern "C" int nsa_skinny_linear(int32_t rows, int32_t k, int32_t n, const void* x, int64_t x_row_stride, const void* norm_weight, float eps,
                                 const void* weight, const void* bias, void* y, int64_t y_row_stride, void* stream) {
  using namespace nsa;
  if (rows <= 0 || k <= 0 || n <= 0 || !x || !weight || !y) return NSA_E_ARG;
  const size_t xb = (size_t)rows * (k + 8) * 2;
  if (rows > 32 || (k & 31) || xb > kSkinnyLds) return NSA_E_UNSUPPORTED;
  if ((x_row_stride & 7) || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(norm_weight)) & 15))
    return NSA_E_ARG;
  const int nb = rows <= 16 ? 1 : 2;
  const size_t shm = sizeof(float) * kSkinnyWaves * nb * 16 * 17 + xb;
  const dim3 grid((unsigned)((n + 15) / 16)), block(kSkinnyThreads);
  hipStream_t st = (hipStream_t)stream;
#define NSA_SKINNY(NB)                                                                                                                           \
  hipLaunchKernelGGL((skinny_linear_kernel<NB>), grid, block, shm, st, rows, k, n, (const __bf16*)x, (long)x_row_stride, (const __bf16*)norm_weight, \
                     eps, (const __bf16*)weight, (const __bf16*)bias, (__bf16*)y, (long)y_row_stride)
  if (nb == 1) NSA_SKINNY(1); else NSA_SKINNY(2);
#undef NSA_SKINNY
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}
