// dK / dV of sliding and compressed attention at 128 features (included by nsa_dense.hip, whose ranges and work distribution it uses):
// one wave per tile of 32 rows, four waves per 64 keys.
//
// dense_bwd_dkv_pipe_kernel shares a tile between two waves, 32 keys each: every operand of Q^T and dO^T read from LDS feeds one
// product, the scores' operands are read twice, and a barrier a tile keeps the waves in step (2400 cycles for 1024 of MFMA a wave).
// Here a wave holds dK and dV of all 64 keys in accumulation registers and takes every fourth tile of the work-group's queries by itself,
// as in the selection's walk (nsa_select_bwd_block.hpp): no barrier in the loop, two products an operand, rows by DMA (Q one tile ahead,
// dO two).  What bounds it is the order of one wave's instructions: 64 products are 2048 cycles, and behind each there is time for about
// six others.  Laid out in slots of one product with its share of the reads, requests, exponentials and conversions a tile takes 2590
// cycles; with the same work in pairs of products, scalars of the next tile at the loop's top and p, dS converted eight at a time, 3100.
// The factors -lse log2e and -delta come ready from the dQ kernel.  Before the loop 6000 - 8000 cycles (latency of the first rows), behind
// it 6700 (four waves' sums through LDS): few work-groups with long chunks of queries.
//
// dQ + dK / dV + their reduction of 32 / 8 heads, us, before (the pipelined walk) and with this one:
//   compressed (stride 16)  4096 tokens 138 -> 122, 8192 300 -> 260, 16384 800 -> 658, 32768 2420 -> 2020
//   sliding (window 512)    4096 tokens 255 -> 186, 8192 405 -> 358, 32768 1450 -> 1340
#pragma once
#include "nsa_pipe.hpp"

namespace nsa {

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1))) void dense_bwd_dkv_keys_kernel(const DensePlan P, const __bf16* __restrict__ q, const __bf16* __restrict__ k,
                                                                                                         const __bf16* __restrict__ v, const __bf16* __restrict__ dout,
                                                                                                         const float* __restrict__ delta, float* __restrict__ part) {
  constexpr int D = 128, KS = D / 16, DT = D / 32, NW = 4, KT = 2;
  constexpr int CPR = D / 8, RPI = 64 / CPR, NT = 32 / RPI;
  constexpr int GB = 1024 + 16, TB = (NT * GB + 255) / 256 * 256, BUFB = 2 * TB;
  __shared__ __align__(1024) char tile_s[NW * 2 * BUFB];        // [wave][tile % 2][Q tile | dO tile]
  __shared__ __align__(16) char kb_s[2 * TB];                  // the K rows
  __shared__ __align__(16) float scal_s[NW][2][64];            // [wave][tile % 2] -lse log2e of the tile's rows, then -delta
  __shared__ __align__(16) int lo_s[NW][32], span_s[NW][32];   // visible rows of k / v, of a tile that needs them
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, n_ = lane & 31, h = lane >> 5;
  const int bh = blockIdx.y, b = bh / P.hkv, hk = bh % P.hkv;
  int T, c, qlo, qhi, c0, c1;
  if (!chunk_of(P, blockIdx.x, T, c, qlo, qhi, c0, c1)) return;
  if (c0 >= c1) return;
  const int lg = P.lg, ppt = 32 >> lg;
  auto tile_off = [](int r, int cc) { return (r / RPI) * GB + (r % RPI) * (2 * D) + 16 * (cc ^ (4 * (r & 3))); };
  typedef __attribute__((address_space(3))) void* lds_p;
  auto lds_addr = [](void* p) { return (unsigned)(unsigned long)(lds_p)p; };
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_addr(tile_s + wave * 2 * BUFB));
  const unsigned scal0 = __builtin_amdgcn_readfirstlane(lds_addr(&scal_s[wave][0][0]));
  const unsigned kbase = __builtin_amdgcn_readfirstlane(lds_addr(kb_s));

  // rows of a tile by buffer loads: a descriptor from the tile's first query on, a lane's own offset from it.  Rows from c1 on are masked;
  // those behind the sequence repeat its last query (see last_rows).
  const int lrow = lane / CPR, pos = lane % CPR;
  const unsigned long qa = (unsigned long)(q + b * P.sq[0] + (long)(hk * P.g) * P.sq[1]), ga = (unsigned long)(dout + b * P.sdo[0] + (long)(hk * P.g) * P.sdo[1]);
  const unsigned q_bytes = 2u * (unsigned)((P.g - 1) * P.sq[1] + (P.n - 1) * P.sq[2] + D), g_bytes = 2u * (unsigned)((P.g - 1) * P.sdo[1] + (P.n - 1) * P.sdo[2] + D);
  const unsigned sqn = 2u * (unsigned)P.sq[2], sgn = 2u * (unsigned)P.sdo[2];
  unsigned qoff[NT], goff[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int rr = t * RPI + lrow;
    const unsigned chunk = 16u * (unsigned)(pos ^ (4 * (lrow & 3)));
    qoff[t] = 2u * (unsigned)(rr & (P.g - 1)) * (unsigned)P.sq[1] + (unsigned)(rr >> lg) * sqn + chunk;
    goff[t] = 2u * (unsigned)(rr & (P.g - 1)) * (unsigned)P.sdo[1] + (unsigned)(rr >> lg) * sgn + chunk;
  }
  // rows from query i on, none where there is no tile
  auto rows_from = [&](unsigned long a, unsigned bytes, unsigned per_query, int i) {
    const unsigned first = (unsigned)i * per_query;
    const unsigned long at = a + (i < c1 ? first : 0u);
    rsrc4 r;
    r[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)at); r[1] = __builtin_amdgcn_readfirstlane((int)(unsigned)(at >> 32));
    r[2] = __builtin_amdgcn_readfirstlane((int)(i < c1 ? bytes - first : 0u)); r[3] = 0x00020000;
    return r;
  };
  // the tile that ends behind the sequence is its wave's last one: its offsets are changed in place
  const int stride = NW * ppt, first = c0 + wave * ppt;
  const int tail = first < c1 ? first + (c1 - 1 - first) / stride * stride : P.n, tail_at = tail + ppt > P.n ? tail : -1;
  auto last_rows = [&](unsigned* off, unsigned per_query) {
    unsigned l = lrow;
    opaque(l);
#pragma unroll
    for (int t = 0; t < NT; ++t) off[t] -= (unsigned)max(0, (int)((t * RPI + l) >> lg) - (P.n - 1 - tail_at)) * per_query;
  };
  auto dma = [&](unsigned dst, unsigned at, rsrc4 rows, auto tc) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(dst), "v"(at), "s"(rows), "n"(decltype(tc)::value * GB) : "memory", "m0", "scc");
  };
  const float* const scal_base = delta + ((size_t)(h ? 0 : gridDim.y) * P.g + (size_t)bh * P.g + (n_ & (P.g - 1))) * P.n;
  auto dma_scal = [&](int i0, int bf) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" :: "s"(scal0 + bf * 256), "v"(scal_base + min(i0 + (n_ >> lg), P.n - 1)) : "memory", "m0");
  };

  // LDS byte addresses of this lane, all of the buffer in use
  constexpr int NR = KS / 2;
  unsigned row_a[NR], krow_a[NR], tr_a[DT], scal_a = scal0 + 16 * h;
  {
    const int ll = lane & 15, e = ll >> 2, qq = ll & 3, mh = (lane >> 4) & 1;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const unsigned o = tile_off(n_, 4 * i + h);
      row_a[i] = lds0 + o; krow_a[i] = kbase + o;
      opaque(row_a[i]); opaque(krow_a[i]);
    }
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      tr_a[i] = lds0 + tile_off(4 * h + e, 4 * i + 2 * mh + (qq >> 1)) + 8 * (qq & 1);
      opaque(tr_a[i]);
    }
    opaque(scal_a);
  }

  int i0 = first;                          // first query of the wave's tile
  auto q_of = [&](int i) { return rows_from(qa, q_bytes, sqn, i); };
  auto g_of = [&](int i) { return rows_from(ga, g_bytes, sgn, i); };
  // Before the loop: V and K rows (a quarter of them a wave; V where the second tile's Q rows will be, until every wave has its operands),
  // Q and dO rows of the first tile, dO rows of the second.  (Operands of V straight from memory, 16 bytes of 32 rows a load: 3000 cycles
  // more a work-group.)
  {
    const int here = min(64, P.krows - kBK * T);
    auto keys_of = [&](const __bf16* x, const long* s) {
      const unsigned long at = (unsigned long)(x + b * s[0] + hk * s[1] + (long)kBK * T * s[2]);
      rsrc4 r;
      r[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)at); r[1] = __builtin_amdgcn_readfirstlane((int)(unsigned)(at >> 32));
      r[2] = __builtin_amdgcn_readfirstlane((int)(2u * ((unsigned)(here - 1) * (unsigned)s[2] + D))); r[3] = 0x00020000;
      return r;
    };
    if (first == tail_at) last_rows(qoff, sqn);
    if (first == tail_at) last_rows(goff, sgn);
    const rsrc4 rv = keys_of(v, P.sv), rk = keys_of(k, P.sk), r0 = q_of(first), r1 = g_of(first), r2 = g_of(first + stride);
    unsigned voff[4], koff[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const unsigned row = 16 * wave + t * RPI + lrow, chunk = 16u * (unsigned)(pos ^ (4 * (lrow & 3)));
      voff[t] = row * 2u * (unsigned)P.sv[2] + chunk; koff[t] = row * 2u * (unsigned)P.sk[2] + chunk;
    }
    fence();
    asm volatile("s_nop 4" ::: "memory");      // (a scalar that a vector instruction wrote may be an address five wait states later)
    static_for<4>([&](auto tc) { dma(lds0 + BUFB, voff[decltype(tc)::value], rv, tc); });
    static_for<4>([&](auto tc) { dma(kbase + 4 * wave * GB, koff[decltype(tc)::value], rk, tc); });
    dma_scal(first, 0);
    static_for<NT>([&](auto tc) { dma(lds0, qoff[decltype(tc)::value], r0, tc); });
    static_for<NT>([&](auto tc) { dma(lds0 + TB, goff[decltype(tc)::value], r1, tc); });
    fence();
    if (first + stride == tail_at) last_rows(goff, sgn);
    static_for<NT>([&](auto tc) { dma(lds0 + BUFB + TB, goff[decltype(tc)::value], r2, tc); });
    fence();
  }
  bf16x8 Vf[KT][KS];
  floatx16 dKa[DT][KT], dVa[DT][KT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) { dKa[dt][kt] = zero_acc(); dVa[dt][kt] = zero_acc(); }
  wait_vm<3 * NT + 1>();
  __syncthreads();
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int row = 32 * kt + n_;
      Vf[kt][ks] = *reinterpret_cast<const bf16x8*>(tile_s + (row >> 4) * 2 * BUFB + BUFB + tile_off(row & 15, 2 * ks + h));
    }
  __syncthreads();

  // queries that see every key of the tile: in [all_lo, all_hi]
  int all_lo = 0, all_hi = c1 - 1;
  {
    const long last = (long)kBK * T + kBK - 1;      // the tile's last row of k / v
    if (last >= P.krows) all_lo = INT_MAX;
    else if (P.mode == 0) { all_lo = (int)max(0l, last - P.wf); all_hi = (int)min((long)all_hi, (long)kBK * T + P.wb); }
    else if (P.causal) all_lo = (int)min((long)INT_MAX, max(0l, (last - P.mem + 1) * P.st));
  }

  const float sc = P.scale * kLog2e;
  int buf = 0, flip = BUFB;
  constexpr int AH = 4, RING = AH + 3;
  constexpr int mB = 2 * KS, mC = 4 * KS, mD = mC + 4 * DT, mN = mD + 4 * DT;      // first MFMA of each run: S, dP, dV, dK
  constexpr int rB = 3 * KS, rC = 4 * KS, rD = rC + 2 * DT, rN = rD + 2 * DT;         // first operand of each run
  rsrc4 rq = q_of(i0 + stride), rg = g_of(i0 + 2 * stride);
  bf16x8 ahead[AH + 2];
  auto request_ahead = [&](unsigned to, auto half) {      // the first operands of the scores, half of them a time
    constexpr int H = (AH + 2) / 2;
    static_for<H>([&](auto ic) {
      constexpr int i = H * decltype(half)::value + decltype(ic)::value, ks = i / 3, w = i % 3;
      if constexpr (w == 0) ahead[i] = lds_read8(row_a[ks / 2] + to + (ks % 2) * 32);
      else ahead[i] = lds_read8(krow_a[ks / 2] + (ks % 2) * 32 + (w - 1) * (32 / RPI * GB));
    });
  };
  wait_vm<NT>();      // (the loop's own wait for dO rows counts on two tiles before it)
  request_ahead(0u, std::integral_constant<int, 0>{});
  request_ahead(0u, std::integral_constant<int, 1>{});
  for (; i0 < c1; i0 += stride) {
    i0 = __builtin_amdgcn_readfirstlane(i0);
    const unsigned cur0 = lds0 + buf * BUFB, other0 = lds0 + (buf ^ 1) * BUFB;
    const int inext = i0 + stride;
    if (inext == tail_at) last_rows(qoff, sqn);
    if (inext + stride == tail_at) last_rows(goff, sgn);
    const bool masked = i0 < all_lo || i0 + ppt - 1 > all_hi;

    floatx16 Sa[KT], Pa[KT], nd;
    floatx4 ls[4];
    unsigned Pw[KT][2][4], Sw[KT][2][4];      // p and dS as bf16, two elements a word
    bf16x8 ring[RING];
    auto rd = [&](auto ic) -> bf16x8 {
      constexpr int i = decltype(ic)::value;
      constexpr unsigned S2 = 8 / RPI * GB, H2 = 16 / RPI * GB, K2 = 32 / RPI * GB;      // 8, 16, 32 rows on
      if constexpr (i < rB) {
        constexpr int ks = i / 3, w = i % 3;
        if constexpr (w == 0) return lds_read8(row_a[ks / 2] + (ks % 2) * 32);
        else return lds_read8(krow_a[ks / 2] + (ks % 2) * 32 + (w - 1) * K2);
      } else if constexpr (i < rC) return lds_read8(row_a[(i - rB) / 2] + ((i - rB) % 2) * 32 + TB);
      else {
        constexpr bool isq = i >= rD;
        constexpr int j = isq ? i - rD : i - rC, rh = j / DT, dt = j % DT;
        return lds_read8_tr(tr_a[dt] + rh * H2 + (isq ? 0 : TB), tr_a[dt] + rh * H2 + (isq ? 0 : TB) + S2);
      }
    };
    auto need = [](int m) constexpr { return m < mB ? 3 * (m / 2) + 1 + (m & 1) : m < mC ? rB + (m - mB) / 2 : m < mD ? rC + (m - mC) / 2 : rD + (m - mD) / 2; };
    auto upto = [need](int m) constexpr { const int x = need(m) + AH; return x < rN ? x : rN - 1; };
    auto operand = [](const unsigned* w) { return __builtin_bit_cast(bf16x8, (intx4){(int)w[0], (int)w[1], (int)w[2], (int)w[3]}); };
    // (the words are opaque: the compiler would convert all eight elements right before the product that takes them)
    auto pair = [](float x, float y) {
      typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
      unsigned w = __builtin_bit_cast(unsigned, (bf16x2){(__bf16)x, (__bf16)y});
      opaque(w);
      return w;
    };
    auto exps = [&](int x) {      // elements in pairs of rows, the two halves of the keys in turn
      const int kt = (x >> 1) & 1, e = (x >> 2) * 2 + (x & 1);
      Sa[kt][e] = fast_exp2(__builtin_fmaf(Sa[kt][e], sc, ls[e >> 2][e & 3]));
      if (e & 1) Pw[kt][e >> 3][(e & 7) >> 1] = pair(Sa[kt][e - 1], Sa[kt][e]);
    };
    auto dss2 = [&](int x) {
      const int kt = x & 1, e = (x >> 1) * 2;
      Sw[kt][e >> 3][(e & 7) >> 1] = pair(Sa[kt][e] * Pa[kt][e], Sa[kt][e + 1] * Pa[kt][e + 1]);
    };

    static_for<AH + 2>([&](auto ic) { ring[decltype(ic)::value % RING] = ahead[decltype(ic)::value]; });
    // slot m: product m, and behind it what it leaves time for (about six instructions, an exponential counts for two)
    static_for<mN>([&](auto mc) {
      constexpr int m = decltype(mc)::value, i = need(m), kt = m & 1;
      if constexpr (m < mB) {
        constexpr int ks = m / 2;
        Sa[kt] = mfma32(ring[(3 * ks) % RING], ring[i % RING], ks == 0 ? zero_acc() : Sa[kt]);
      } else if constexpr (m < mC) {
        constexpr int ks = (m - mB) / 2;
        Pa[kt] = mfma32(ring[i % RING], Vf[kt][ks], ks == 0 ? nd : Pa[kt]);
      } else {
        constexpr int c0_ = (m < mD ? m - mC : m - mD) / 2, rh = c0_ / DT, dt = c0_ % DT;
        if constexpr (m < mD) mfma32_acc<c0_ % DT == 0>(dVa[dt][kt], ring[i % RING], operand(Pw[kt][rh]));
        else mfma32_acc<c0_ % DT == 0>(dKa[dt][kt], ring[i % RING], operand(Sw[kt][rh]));
      }
      fence();
      if constexpr (m + 1 < mN) {
        constexpr int lo = upto(m) + 1, hi = upto(m + 1);
        if constexpr (hi >= rB && lo <= rB) {      // dO rows: asked for two tiles ago, behind them this tile's Q, the next one's dO and so many ...
          constexpr int issued = (m > 1) + (m < 3 ? 0 : ((m < 15 ? m : 15) - 1) / 2) + (m > 15);      // ... of the next one's Q
          wait_vm<2 * NT + 1 + issued>();
          fence();
        }
        if constexpr (hi >= lo) static_for<hi - lo + 1>([&](auto jc) {
          constexpr int j = lo + decltype(jc)::value;
          ring[j % RING] = rd(std::integral_constant<int, j>{});
        });
      }
      if constexpr (m < mB) {
        if constexpr (m == 1) dma_scal(inext, buf ^ 1);
        if constexpr (m >= 2 && (m & 1) == 0) dma(other0, qoff[m / 2 - 1], rq, std::integral_constant<int, m / 2 - 1>{});
        if constexpr (m == mB - 1) dma(other0, qoff[NT - 1], rq, std::integral_constant<int, NT - 1>{});
        if constexpr (m >= mB - 7 && m < mB - 3) {
          constexpr int a = m - (mB - 7);
          const floatx4 d4 = *(lds_f4)(scal_a + 128 + 32 * a);
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) nd[4 * a + bb] = d4[bb];
        }
        if constexpr (m == mB - 2) ls[0] = *(lds_f4)(scal_a);
      } else if constexpr (m < mC) {
        constexpr int s = m - mB;
        if constexpr (s == 1 || s == 5 || s == 9) ls[(s + 3) / 4] = *(lds_f4)(scal_a + 32 * ((s + 3) / 4));
        static_for<(3 * (s + 1)) / 2 - (3 * s) / 2>([&](auto jc) { exps((3 * s) / 2 + decltype(jc)::value); });      // three in two slots
      } else if constexpr (m < mD) {
        constexpr int s = m - mC;
        if constexpr (s < 2 * DT) exps(24 + s);
        else dss2(s - 2 * DT);
      } else {
        constexpr int s = m - mD;
        if constexpr (s < 2 * DT) dss2(s + 2 * DT);
        if constexpr (s < 8 ? (s & 1) == 0 : s < 12) {      // over the dO rows, which nothing reads any more
          constexpr int t = s < 8 ? s / 2 : s - 4;
          dma(cur0 + TB, goff[t], rg, std::integral_constant<int, t>{});
        }
        if constexpr (s == 12) { wait_vm<NT>(); request_ahead((unsigned)flip, std::integral_constant<int, 0>{}); }      // Q rows and scalars: asked for a tile ago
        if constexpr (s == 13) { request_ahead((unsigned)flip, std::integral_constant<int, 1>{}); rq = q_of(inext + stride); }
        if constexpr (s == 14) rg = g_of(inext + 2 * stride);
      }
      fence();
      if constexpr (m == mB - 1) {
        if (masked) {      // row r sees keys lo .. lo + span; a row that is not there has a lo behind all keys
          if (h == 0) {
            const int i = i0 + (n_ >> lg);
            const Interval me = visible_range(P, min(i, P.n - 1));
            const int lo = P.mode == 0 ? me.lo : 0, hi = P.mode == 0 ? me.hi : me.hi + P.mem;
            lo_s[wave][n_] = i >= c1 || hi < lo ? INT_MAX : lo;
            span_s[wave][n_] = max(hi - lo, 0);
          }
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const intx4 l4 = *reinterpret_cast<const intx4*>(&lo_s[wave][8 * a + 4 * h]), s4 = *reinterpret_cast<const intx4*>(&span_s[wave][8 * a + 4 * h]);
#pragma unroll
            for (int bb = 0; bb < 4; ++bb) {
              const unsigned at = (unsigned)(kBK * T + n_ - l4[bb]);
#pragma unroll
              for (int kt = 0; kt < KT; ++kt) Sa[kt][4 * a + bb] = at + 32 * kt <= (unsigned)s4[bb] ? Sa[kt][4 * a + bb] : -INFINITY;
            }
            fence();
          }
        }
        fence();
      }
    });
#pragma unroll
    for (int i = 0; i < NR; ++i) row_a[i] += flip;
#pragma unroll
    for (int i = 0; i < DT; ++i) tr_a[i] += flip;
    scal_a += buf ? -256 : 256;
    flip = -flip;
    buf ^= 1;
  }

  // the four waves' sums, a tensor at a time: float4 chunk cc of key row kl at cc ^ (kl % chunks)
  wait_vm<0>();
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // the last MFMAs have written their results
  fence();
  constexpr int FPR = D / 4;
  floatx4* red = reinterpret_cast<floatx4*>(tile_s);
  float* dst = part + (((size_t)bh * P.key_tiles + T) * P.chunks + c) * (2 * kBK * D);
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    __syncthreads();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          floatx4 x;
#pragma unroll
          for (int bb = 0; bb < 4; ++bb) x[bb] = which == 0 ? dKa[dt][kt][4 * a + bb] : dVa[dt][kt][4 * a + bb];
          const int kl = 32 * kt + n_, cc = 8 * dt + 2 * a + h;
          red[(wave * 64 + kl) * FPR + (cc ^ (kl & (FPR - 1)))] = x;
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * FPR / 256; ++i) {
      const int e = threadIdx.x + 256 * i, kl = e / FPR, cc = e % FPR, p = kl * FPR + (cc ^ (kl & (FPR - 1)));
      floatx4 s = red[p];
#pragma unroll
      for (int w = 1; w < NW; ++w) s += red[w * 64 * FPR + p];
      *reinterpret_cast<floatx4*>(dst + which * kBK * D + (size_t)kl * D + 4 * cc) = s;
    }
  }
}

}  // namespace nsa
