// Projections of a decode step: y = norm(x) W^T + bias for a handful of rows (one token per sequence, NSA.py:356-364, 545), with
// the RMS norm in front (NSA.py:230) when asked for.
//
// Bound by reading W once: 2 K N bytes.  A work-group of eight waves owns 16 output features and shares the K axis, so 4096
// features are 2048 waves that each request up to 16 KB of W before waiting for the first; the batch is the other side of a
// 16x16x32 MFMA.  While W is on its way the work-group brings x into LDS and norms it there - the norm costs no launch and
// no pass of its own.  The waves' partial sums meet in LDS; bias, activation and residual are added there, each rounded to
// bf16 as the layers they replace would (a decode step of a small model is bound by the number of its launches).
// Measured (weights from HBM, launch included): 4096 -> 6240 with norm, batch 1 14.5 us, batch 8 18.1 us, of which the 51 MB
// of W take 9.8 us at the rate of a large copy (norm kernel + library GEMM: 20.6 / 20.8 us); 4096 -> 4096, batch 1 10.2 us (15.6 us);
// 1024 -> 1584 with norm, batch 16 6.4 us (9.3 us).
#include "nsa_common.hpp"
#include "../../include/nsa_hip.h"

namespace nsa {

constexpr int kSkinnyWaves = 8, kSkinnyThreads = 64 * kSkinnyWaves;
constexpr int kSkinnyAhead = 16;                 // K steps (of 32) whose W operands a wave holds
constexpr size_t kSkinnyLds = 128 << 10;         // of x

struct SkinnyArgs {
  int rows, K;
  const __bf16* x;
  long xs;
  const __bf16* nw;                // norm weight or null
  float eps;
  int tiles0;                      // work-groups of output 0; the rest are output 1's
  int n[2];
  const __bf16 *w[2], *bias[2];
  __bf16* y[2];
  long ys[2];
  int act;                         // NSA_ACT_*
  const __bf16* res;               // added to output 0, or null
  long rs;
};

// NB: groups of 16 rows
template <int NB>
__global__ __launch_bounds__(kSkinnyThreads, 4) void skinny_linear_kernel(const SkinnyArgs A) {
  extern __shared__ __align__(16) char lds[];
  __shared__ float ss_s[kSkinnyWaves];
  float (*part_s)[NB][16][17] = reinterpret_cast<float (*)[NB][16][17]>(lds);                                 // [wave]
  __bf16* x_s = reinterpret_cast<__bf16*>(lds + sizeof(float) * kSkinnyWaves * NB * 16 * 17);
  const int o = (int)blockIdx.x < A.tiles0 ? 0 : 1;
  const int rows = A.rows, K = A.K, N = A.n[o];
  const __bf16* __restrict__ x = A.x;
  const __bf16* __restrict__ nw = A.nw;
  const __bf16* __restrict__ w = A.w[o];
  const long xs = A.xs;
  const float eps = A.eps;
  const int RS = K + 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, kq = lane >> 4;
  const int n0 = ((int)blockIdx.x - (o ? A.tiles0 : 0)) * 16;
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
      for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
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
    if (A.bias[o] != nullptr) t += (float)A.bias[o][n0 + f];
    const int row = 16 * g + br;
    if (A.act == NSA_ACT_GELU) {
      const float u = (float)(__bf16)t;
      t = 0.5f * u * (1.0f + erff(u * 0.70710678118654752f));
    } else if (A.act == NSA_ACT_RELU) {
      t = t < 0.f ? 0.f : t;                              // (NaN stays, as the layer leaves it)
    }
    if (o == 0 && A.res != nullptr) t = (float)(__bf16)t + (float)A.res[row * A.rs + n0 + f];
    A.y[o][row * A.ys[o] + n0 + f] = (__bf16)t;
  }
}

static int launch_skinny(const SkinnyArgs& A, void* stream) {
  if (A.rows <= 0 || A.K <= 0 || A.n[0] <= 0 || A.n[1] < 0 || !A.x || !A.w[0] || !A.y[0] || (A.n[1] > 0 && (!A.w[1] || !A.y[1]))) return NSA_E_ARG;
  const size_t xb = (size_t)A.rows * (A.K + 8) * 2;
  if (A.rows > 32 || (A.K & 31) || xb > kSkinnyLds) return NSA_E_UNSUPPORTED;
  if ((A.xs & 7) || ((reinterpret_cast<uintptr_t>(A.x) | reinterpret_cast<uintptr_t>(A.w[0]) | reinterpret_cast<uintptr_t>(A.w[1]) |
                      reinterpret_cast<uintptr_t>(A.nw)) & 15))
    return NSA_E_ARG;
  const int nb = A.rows <= 16 ? 1 : 2;
  const size_t shm = sizeof(float) * kSkinnyWaves * nb * 16 * 17 + xb;
  const dim3 grid((unsigned)(A.tiles0 + (A.n[1] + 15) / 16)), block(kSkinnyThreads);
  hipStream_t st = (hipStream_t)stream;
  if (nb == 1) hipLaunchKernelGGL((skinny_linear_kernel<1>), grid, block, shm, st, A);
  else hipLaunchKernelGGL((skinny_linear_kernel<2>), grid, block, shm, st, A);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

}  // namespace nsa

extern "C" int nsa_skinny_linear(int32_t rows, int32_t k, int32_t n, const void* x, int64_t x_row_stride, const void* norm_weight, float eps,
                                 const void* weight, const void* bias, int32_t act, const void* residual, int64_t residual_row_stride, void* y,
                                 int64_t y_row_stride, void* stream) {
  using namespace nsa;
  if (act < NSA_ACT_NONE || act > NSA_ACT_RELU) return NSA_E_ARG;
  SkinnyArgs A{};
  A.rows = rows; A.K = k; A.x = (const __bf16*)x; A.xs = x_row_stride; A.nw = (const __bf16*)norm_weight; A.eps = eps;
  A.tiles0 = (n + 15) / 16; A.n[0] = n; A.w[0] = (const __bf16*)weight; A.bias[0] = (const __bf16*)bias; A.y[0] = (__bf16*)y; A.ys[0] = y_row_stride;
  A.act = act; A.res = (const __bf16*)residual; A.rs = residual_row_stride;
  return launch_skinny(A, stream);
}

// ---------------------------------------------------------------------------- few rows in fp32
// y = act(x W^T + bias) for matrices too small for the GEMM library's tiles (an fp32 layer on a few dozen tokens: 240 x 256 x
// 256 takes it 65 us, one 256 x 256 tile and seven eighths of it idle).  A work-group owns a 32 x 32 tile of y and its eight waves
// share K: v_mfma_f32_32x32x2, both operands 16 bytes per lane straight from memory (lane = row, half h: features
// 8 t + 4 h + j in step j of group t), partial tiles added in LDS in a fixed order.
// A layer on a few tokens is bound by its launches, so what stands beside a projection goes into its launch: a second projection (of
// the same input, or of another of the same sizes), the RMS norm of the input - its weight is multiplied in on the way, its factor is
// one per row and applied to the finished sums - and the strategy gate over three attention branches in front of the output
// projection.  The usage example of the package (2 x 31 tokens of 512 features): 17 launches
// and 334 us -> 8 and 215.

namespace nsa {

struct LinearF32Part { const float *x, *w, *bias; float* y; int n; };
struct LinearF32Args {
  LinearF32Part p[2];
  int rows, K, tiles0, act;        // tiles0: work-groups along x of part 0
  long xs;
  int norm;
  const float* nw;                 // norm weight, or null for ones
  float eps;
  // gate: x is sum_t sigmoid(logits[row, 3 head + t]) branch_t[b, head, i], feature head * d + f of row b n + i
  const float *logits, *branch[3];
  long sb[3][3];
  int seq, d, heads;
};

template <bool GATED>
__global__ __launch_bounds__(512) void linear_f32_kernel(const LinearF32Args A) {
  __shared__ float part_s[8][32][33];
  __shared__ float ss_s[8][2][32];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, h = lane >> 5;
  const bool second = (int)blockIdx.x >= A.tiles0;
  const LinearF32Part P = second ? A.p[1] : A.p[0];
  const int rows = A.rows, K = A.K, N = P.n;
  const int n0 = ((int)blockIdx.x - (second ? A.tiles0 : 0)) * 32, m0 = blockIdx.y * 32;
  const int groups = K >> 3, per = (groups + 7) / 8, g0 = wave * per, g1 = min(groups, g0 + per);
  const float* wp = P.w + (long)min(n0 + r, N - 1) * K + 4 * h;
  const int row = min(m0 + r, rows - 1);
  floatx16 acc = zero_acc();
  auto products = [&](floatx4 a, floatx4 b) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], acc, 0, 0, 0);
  };
  if constexpr (GATED) {
    const int bb = row / A.seq, i = row - bb * A.seq;
    const float* lp = A.logits + (long)row * 3 * A.heads;
    const float* bp[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) bp[t] = A.branch[t] + bb * A.sb[t][0] + (long)i * A.sb[t][2];
#pragma unroll 2
    for (int g = g0; g < g1; ++g) {
      const int f = 8 * g + 4 * h, head = f / A.d, at = f - head * A.d;
      floatx4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < 3; ++t) x += *reinterpret_cast<const floatx4*>(bp[t] + (long)head * A.sb[t][1] + at) * (1.f / (1.f + expf(-lp[3 * head + t])));
      products(*reinterpret_cast<const floatx4*>(wp + 8 * g), x);
    }
  } else {
    const float* xp = P.x + (long)row * A.xs + 4 * h;
    if (!A.norm) {
#pragma unroll 4
      for (int g = g0; g < g1; ++g) products(*reinterpret_cast<const floatx4*>(wp + 8 * g), *reinterpret_cast<const floatx4*>(xp + 8 * g));
    } else {
      const float* np = A.nw + 4 * h;
      float ss = 0.f;
#pragma unroll 4
      for (int g = g0; g < g1; ++g) {
        const floatx4 x = *reinterpret_cast<const floatx4*>(xp + 8 * g);
        // (a feature that is not finite makes the row's norm NaN; squares that overflow make it infinite and the normed row zero)
        ss += (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = __builtin_fmaf(x[e], 0.f, ss);
        products(*reinterpret_cast<const floatx4*>(wp + 8 * g), A.nw != nullptr ? x * *reinterpret_cast<const floatx4*>(np + 8 * g) : x);
      }
      ss_s[wave][h][r] = ss;
    }
  }
  // D: feature 8 (i / 4) + 4 h + i % 4, row r
#pragma unroll
  for (int i = 0; i < 16; ++i) part_s[wave][r][8 * (i / 4) + 4 * h + (i % 4)] = acc[i];
  __syncthreads();
  for (int e = threadIdx.x; e < 1024; e += 512) {
    const int f = e & 31, mr = e >> 5;
    if (m0 + mr >= rows || n0 + f >= N) continue;
    float t = 0.f;
#pragma unroll
    for (int v = 0; v < 8; ++v) t += part_s[v][mr][f];
    if (!GATED && A.norm) {
      float ss = 0.f;
#pragma unroll
      for (int v = 0; v < 8; ++v) ss += ss_s[v][0][mr] + ss_s[v][1][mr];
      const float rs = rsqrtf(ss / (float)K + A.eps);
      t = rs == 0.f ? 0.f : t * rs;
    }
    if (P.bias != nullptr) t += P.bias[n0 + f];
    if (A.act == NSA_ACT_RELU) t = t < 0.f ? 0.f : t;      // (NaN stays)
    P.y[(long)(m0 + mr) * N + n0 + f] = t;
  }
}

// what the kernel takes for granted of its two parts
static int check_linear_f32(const LinearF32Args& A) {
  if (A.rows <= 0 || A.K <= 0 || (A.act != NSA_ACT_NONE && A.act != NSA_ACT_RELU)) return NSA_E_ARG;
  if ((A.K & 7) || (A.rows + 31) / 32 > 65535) return NSA_E_UNSUPPORTED;
  for (const LinearF32Part& P : A.p) {
    if (P.n < 0 || (P.n > 0 && (!P.w || !P.y)) || (reinterpret_cast<uintptr_t>(P.x) | reinterpret_cast<uintptr_t>(P.w)) & 15) return NSA_E_ARG;
  }
  return A.p[0].n <= 0 || (A.xs & 3) || reinterpret_cast<uintptr_t>(A.nw) & 15 ? NSA_E_ARG : 0;
}

template <bool GATED>
static int launch_linear_f32(LinearF32Args& A, void* stream) {
  if (int e = check_linear_f32(A)) return e;
  A.tiles0 = (A.p[0].n + 31) / 32;
  const dim3 grid((unsigned)(A.tiles0 + (A.p[1].n + 31) / 32), (unsigned)((A.rows + 31) / 32));
  hipLaunchKernelGGL(linear_f32_kernel<GATED>, grid, dim3(512), 0, (hipStream_t)stream, A);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

}  // namespace nsa

extern "C" int nsa_linear_f32(int32_t rows, int32_t k, int32_t n, const float* x, int64_t x_row_stride, const float* weight, const float* bias,
                              int32_t act, float* y, void* stream) {
  using namespace nsa;
  if (!x || n <= 0) return NSA_E_ARG;
  LinearF32Args A{};
  A.p[0] = LinearF32Part{x, weight, bias, y, n};
  A.rows = rows; A.K = k; A.xs = (long)x_row_stride; A.act = act;
  return launch_linear_f32<false>(A, stream);
}

extern "C" int nsa_linear_pair_f32(int32_t rows, int32_t k, int64_t x_row_stride, int32_t norm, const float* norm_weight, float eps, int32_t act,
                                   const float* x, const float* weight, const float* bias, int32_t n, float* y, const float* x2, const float* weight2,
                                   const float* bias2, int32_t n2, float* y2, void* stream) {
  using namespace nsa;
  if (!x || !x2 || n <= 0 || n2 <= 0 || (!norm && norm_weight)) return NSA_E_ARG;
  LinearF32Args A{};
  A.p[0] = LinearF32Part{x, weight, bias, y, n};
  A.p[1] = LinearF32Part{x2, weight2, bias2, y2, n2};
  A.rows = rows; A.K = k; A.xs = (long)x_row_stride; A.act = act;
  A.norm = norm ? 1 : 0; A.nw = norm_weight; A.eps = eps;
  return launch_linear_f32<false>(A, stream);
}

extern "C" int nsa_gate_linear_f32(int32_t batch, int32_t heads, int32_t seq, int32_t dim_head, const float* logits, const float* c, const int64_t* c_stride,
                                   const float* f, const int64_t* f_stride, const float* s, const int64_t* s_stride, const float* weight, const float* bias,
                                   int32_t n, float* y, void* stream) {
  using namespace nsa;
  if (!logits || !c || !f || !s || !c_stride || !f_stride || !s_stride || batch <= 0 || heads <= 0 || seq <= 0 || n <= 0) return NSA_E_ARG;
  if (dim_head <= 0 || (dim_head & 3) || (long)batch * seq > 0x7fffffffL || (long)heads * dim_head > 0x7fffffffL) return NSA_E_UNSUPPORTED;
  LinearF32Args A{};
  A.p[0] = LinearF32Part{nullptr, weight, bias, y, n};
  A.rows = batch * seq; A.K = heads * dim_head; A.logits = logits; A.seq = seq; A.d = dim_head; A.heads = heads;
  const float* br[3] = {c, f, s};
  const int64_t* st[3] = {c_stride, f_stride, s_stride};
  for (int t = 0; t < 3; ++t) {
    A.branch[t] = br[t];
    if (reinterpret_cast<uintptr_t>(br[t]) & 15) return NSA_E_ARG;
    for (int e = 0; e < 3; ++e) {
      A.sb[t][e] = (long)st[t][e];
      if (st[t][e] & 3) return NSA_E_ARG;
    }
  }
  return launch_linear_f32<true>(A, stream);
}

// ---------------------------------------------------------------------------- a layer's decode step
// Norm + qkv projection + gate logits (one launch), the attention step (nsa_decode_step: three), output projection + residual:
// one host call, because at small sizes the host's work between the launches is most of the step.

namespace nsa {
// nsa_decode.hip
int run_decode_step(const nsa_decode_step_desc* d, int32_t* state, const void* q, const void* k, const void* v, const void* freqs, int freqs_bf16,
                    void* k_cache, void* v_cache, const void* ck_cache, const void* cv_cache, const void* mem_k, const void* mem_v, void* krun,
                    void* vrun, int64_t krun_row, int64_t vrun_row, int32_t ring, const void* gate_logits, int64_t gate_row, const void* gate_bias,
                    void* ws, size_t ws_bytes, void* out, bool advance, void* stream);

struct LayerLayout { size_t step, off_qkv, off_gate, off_merged, total; };

static int make_layer_layout(const nsa_decode_step_desc* d, LayerLayout& L) {
  if (int e = nsa_decode_step_workspace_bytes(d, &L.step, nullptr, nullptr, nullptr)) return e;
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  L.off_qkv = up(L.step);
  L.off_gate = up(L.off_qkv + (size_t)d->batch * (d->heads + 2 * d->kv_heads) * d->dim_head * 2);
  L.off_merged = up(L.off_gate + (size_t)d->batch * 3 * d->heads * 2);
  L.total = up(L.off_merged + (size_t)d->batch * d->heads * d->dim_head * 2);
  return 0;
}
}  // namespace nsa

extern "C" int nsa_decode_layer_workspace_bytes(const nsa_decode_step_desc* desc, size_t* bytes) {
  nsa::LayerLayout L;
  if (!desc || !bytes) return NSA_E_ARG;
  if (int e = nsa::make_layer_layout(desc, L)) return e;
  *bytes = L.total;
  return 0;
}

extern "C" int nsa_decode_layer(const nsa_decode_step_desc* desc, int32_t dim, const void* x, const void* norm_weight, float eps, const void* w_qkv,
                                const void* w_gate, const void* b_gate, const void* freqs, int32_t freqs_bf16, void* k_cache, void* v_cache, const void* ck_cache,
                                const void* cv_cache, const void* mem_k, const void* mem_v, void* k_run_row, void* v_run_row, const void* w_out,
                                const void* b_out, const void* residual, void* ws, size_t ws_bytes, void* out, void* stream) {
  using namespace nsa;
  if (!desc || !norm_weight || !w_gate || !ws || !out) return NSA_E_ARG;
  LayerLayout L;
  if (int e = make_layer_layout(desc, L)) return e;
  if (ws_bytes < L.total) return NSA_E_WORKSPACE;
  char* w = (char*)ws;
  const int hd = desc->heads * desc->dim_head, kd = desc->kv_heads * desc->dim_head, width = hd + 2 * kd;
  SkinnyArgs P{};
  P.rows = desc->batch; P.K = dim; P.x = (const __bf16*)x; P.xs = dim; P.nw = (const __bf16*)norm_weight; P.eps = eps;
  P.tiles0 = (width + 15) / 16;
  P.n[0] = width; P.w[0] = (const __bf16*)w_qkv; P.y[0] = (__bf16*)(w + L.off_qkv); P.ys[0] = width;
  P.n[1] = 3 * desc->heads; P.w[1] = (const __bf16*)w_gate; P.bias[1] = (const __bf16*)b_gate; P.y[1] = (__bf16*)(w + L.off_gate); P.ys[1] = 3 * desc->heads;
  if (int e = launch_skinny(P, stream)) return e;
  nsa_decode_step_desc d = *desc;
  d.q_stride[0] = d.k_stride[0] = d.v_stride[0] = width;
  d.q_stride[1] = d.k_stride[1] = d.v_stride[1] = desc->dim_head;
  const __bf16* q = (const __bf16*)(w + L.off_qkv);
  if (int e = run_decode_step(&d, nullptr, q, q + hd, q + hd + kd, freqs, freqs_bf16, k_cache, v_cache, ck_cache, cv_cache, mem_k, mem_v, k_run_row,
                              v_run_row, 0, 0, 0, w + L.off_gate, 0, nullptr, ws, L.step, w + L.off_merged, false, stream))
    return e;
  SkinnyArgs O{};
  O.rows = desc->batch; O.K = hd; O.x = (const __bf16*)(w + L.off_merged); O.xs = hd;
  O.tiles0 = (dim + 15) / 16; O.n[0] = dim; O.w[0] = (const __bf16*)w_out; O.bias[0] = (const __bf16*)b_out; O.y[0] = (__bf16*)out; O.ys[0] = dim;
  O.res = (const __bf16*)residual; O.rs = dim;
  return launch_skinny(O, stream);
}
