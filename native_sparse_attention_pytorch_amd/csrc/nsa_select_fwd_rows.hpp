// The forward walk of block-selection attention with its rows gathered by DMA (included by nsa_select.hip, whose unit and list
// helpers it uses): sel_fwd_kernel's work and, but for the order of two roundings, its arithmetic - a wave holds a block's K and V^T
// as operands and streams 32-row tiles.  What bounded that walk were its instructions (seq 32k, 32 / 8 heads, d 128: 1.45 ms, 1.23 with
// the rows cached and no stores).  Here the Q rows go straight into LDS (buffer_load ... lds, two tiles ahead; layout as in
// nsa_select_bwd_block.hpp), which frees the staging registers - two waves a SIMD at 128 features instead of one - and half of the
// loop's instructions; the probabilities go into the products unnormalised, 16 keys behind the exponentials of the next 16, and the
// output rows leave over the Q rows they came from.  Without stores and gathers it takes 0.70 ms now; with them 1.30: the stores
// (4.3 GB of partial rows and their 4-byte lse's, 0.12 ms of it the latter) set the pace.  2048 tokens 77 -> 58 us; d 64, 16 / 4 heads:
// 8192 tokens 86 -> 82 us, 4 x 4096 138 -> 130.
#pragma once
#include "nsa_pipe.hpp"
#include "nsa_select_plan.hpp"

namespace nsa {

// UNI: the rows of a gather instruction are heads of one pair and have one scalar offset
template <int D, int KT, bool UNI>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void sel_fwd_rows_kernel(const SelPlan P, const SmallDiv by_sp, const __bf16* __restrict__ q,
                                                                                                                 const __bf16* __restrict__ k, const __bf16* __restrict__ v,
                                                                                                                 const char* __restrict__ iws, char* __restrict__ fws) {
  constexpr int KS = D / 16, DT = D / 32, CPR = D / 8, RPI = 64 / CPR, NT = 32 / RPI;
  constexpr int GB = 1024 + 16, TB = (NT * GB + 255) / 256 * 256;
  __shared__ __align__(1024) char tile_s[2 * TB];              // [tile % 2] Q rows, later the tile's output rows
  __shared__ __align__(8) char* place_s[2][32];                // where each row's partial goes
  __shared__ int list_s[256];                                   // the unit's pairs
  const int lane = threadIdx.x, n_ = lane & 31, h = lane >> 5;
  int bh, u;
  if (!xcd_map(P, 0, bh, u)) return;
  const int b = bh / P.hkv, hk = bh % P.hkv;
  UnitInfo ui;
  if (!locate_unit(P, iws, 0, bh, u, ui)) return;
  const int lg = P.lg, ppt = 32 >> lg, count = ui.v1 - ui.v0;
  // K, V and the unit's pairs are asked for together
  int pairs[4];
  {
    const int* list = reinterpret_cast<const int*>(iws + P.off_list) + (size_t)bh * P.list_cap;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int pv = ui.v0 + min(lane + 64 * i, count - 1);
      long li = (long)ui.lst0 + max(pv - ui.own, 0);
      li = li < P.list_cap ? li : P.list_cap - 1;
      pairs[i] = list[li];
    }
  }
  bf16x8 Kf[KT][KS], Vraw[KT][DT][2];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    const int kl = 32 * kt + n_;
    const long key = (long)ui.j * P.B + kl;
    const bool ok = kl < P.B && key < P.n;
    const __bf16* kp = k + b * P.sk[0] + hk * P.sk[1] + (ok ? key : 0) * P.sk[2] + 8 * h;
    const __bf16* vp = v + b * P.sv[0] + hk * P.sv[1] + (ok ? key : 0) * P.sv[2] + 8 * h;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) Kf[kt][ks] = ok ? load8(kp + 16 * ks) : zero_frag();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      Vraw[kt][dt][0] = ok ? load8(vp + 32 * dt) : zero_frag();
      Vraw[kt][dt][1] = ok ? load8(vp + 32 * dt + 16) : zero_frag();
    }
  }
  fence();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int pv = ui.v0 + min(lane + 64 * i, count - 1);
    list_s[lane + 64 * i] = pv < ui.own ? (ui.j * P.B + pv) * P.SP + P.S : pairs[i];
  }
  __syncthreads();

  typedef __attribute__((address_space(3))) void* lds_p;
  auto lds_addr = [](void* p) { return (unsigned)(unsigned long)(lds_p)p; };
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_addr(tile_s));
  const int lrow = lane / CPR, pos = lane % CPR;
  auto swz = [](int r) { return D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1) + 2 * ((r >> 2) & 1); };
  auto tile_off = [swz](int r, int c) { return (r / RPI) * GB + (r % RPI) * (2 * D) + 16 * (c ^ swz(r)); };
  const unsigned sqh = 2u * (unsigned)P.sq[1], sqt = 2u * (unsigned)P.sq[2];
  const unsigned vq0 = 16u * (pos ^ swz(lrow)) + (UNI ? (unsigned)lrow * sqh : 0u);
  const unsigned head_q = (unsigned)(n_ & (P.g - 1)) * sqh, head_d = (unsigned)(n_ & (P.g - 1)) * (2 * D);
  const unsigned pair_bytes = (unsigned)P.g * (2 * D);
  char* const opart = fws + P.off_opart + (size_t)bh * P.n * P.SP * pair_bytes;
  char* const spare = fws + P.off_opart + P.prow * (2 * D);
  const unsigned long qa = (unsigned long)(q + b * P.sq[0] + (long)(hk * P.g) * P.sq[1]);
  rsrc4 rows;
  rows[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)qa); rows[1] = __builtin_amdgcn_readfirstlane((int)(unsigned)(qa >> 32)); rows[2] = -1; rows[3] = 0x00020000;
  const float sc = P.scale * kLog2e;

  // tile t: byte offset of this lane's row; leaves the row's place
  auto decode = [&](int t, int raw) {
    const bool live = t * ppt + (n_ >> lg) < count;
    const unsigned qi = __umulhi(2u * (unsigned)raw, by_sp.mul) >> by_sp.sh;
    place_s[t & 1][n_] = live ? opart + (unsigned long)(unsigned)raw * pair_bytes + head_d : spare;
    return qi * sqt + head_q;
  };
  auto pair_of = [&](int t) { return list_s[min(t * ppt + (n_ >> lg), count - 1)]; };
  struct Offsets { int row[NT]; };      // of the gather instructions: scalars where their rows are one pair's, a lane's own otherwise
  auto offsets = [&](unsigned o) {
    Offsets r;
#pragma unroll
    for (int t = 0; t < NT; ++t) r.row[t] = UNI ? __builtin_amdgcn_readlane(o, t * RPI) : __shfl((int)o, t * RPI + lrow, 64) + (int)vq0;
    return r;
  };
  auto gather = [&](const Offsets& o, unsigned dst, auto tc) {
    constexpr int t = decltype(tc)::value;
    const int at = o.row[t];
    if constexpr (UNI && t > 0)
      asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(dst), "v"(vq0), "s"(rows), "s"(at), "n"(t * GB) : "memory", "m0", "scc");
    else if constexpr (UNI)
      asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(dst), "v"(vq0), "s"(rows), "s"(at), "n"(t * GB) : "memory", "m0", "scc");
    else
      asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" :: "s"(dst), "v"(at), "s"(rows), "n"(t * GB) : "memory", "m0", "scc");
  };
  // LDS byte addresses of this lane
  constexpr int RSTEP = KS / 4;
  unsigned row_a[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) { row_a[i] = lds0 + tile_off(n_, 2 * RSTEP * i + h); opaque(row_a[i]); }
  unsigned stw_a = lds0 + 2 * D * n_ + 16 * (n_ & (CPR - 1)) + 8 * h, str_a = lds0 + 2 * D * lrow + 16 * (pos ^ (lrow & (CPR - 1)));
  opaque(stw_a); opaque(str_a);

#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const Offsets o = offsets(decode(t, pair_of(t)));
    fence();
    static_for<NT>([&](auto tc) { gather(o, lds0 + t * TB, tc); });
    fence();
  }
  int raw = pair_of(2);
  bf16x8 VT[DT][KT][2];
  {
    bf16x8 ilo, ihi;
    make_ident(lane, ilo, ihi);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        floatx16 t = mfma32(Vraw[kt][dt][0], ilo, zero_acc());
        t = mfma32(Vraw[kt][dt][1], ihi, t);
        VT[dt][kt][0] = pack8(t, 0);
        VT[dt][kt][1] = pack8(t, 8);
      }
  }
  floatx16 Oa[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) Oa[dt] = zero_acc();
  float lse = 0.f, inv = 0.f;      // of this lane's row of the tile in Oa
  bf16x8 vv[NT];
  char* pr[NT];
  // the tile's output rows over its Q rows: row n_, 16-byte chunk c at position c ^ (n_ % CPR)
  unsigned stw = stw_a, str = str_a;
  auto stage = [&](int c) {
    bf16x4 r;
#pragma unroll
    for (int bb = 0; bb < 4; ++bb) r[bb] = (__bf16)(Oa[c / 4][4 * (c % 4) + bb] * inv);
    *(lds_x4)(stw ^ (unsigned)(16 * c)) = r;
  };
  auto read_rows = [&](int slot, int t) {
    vv[t] = lds_read8((D == 128 ? str ^ (unsigned)(64 * (t & 3)) : str) + t * 1024);
    pr[t] = place_s[slot][t * RPI + lrow];
  };
  auto store_rows = [&](int t) { __builtin_nontemporal_store(vv[t], (glb_x8)(pr[t] + 16 * pos)); };
  auto store_lse = [&](int slot) {
    const unsigned long row = (unsigned long)(place_s[slot][n_] - (fws + P.off_opart)) / (2 * D);
    if (h == 0) reinterpret_cast<float*>(fws + P.off_lsepart)[row] = lse;
  };

  constexpr int AH = 4, RING = AH + 1;
  const int tiles = (count + ppt - 1) / ppt;
  wait_vm<NT>();
  for (int t = 0; t < tiles; ++t) {
    wait_vm<2 * NT>();      // this tile's rows: asked for two tiles ago, behind them a tile's stores and the next tile's rows
    const unsigned cur = (t & 1) * TB;
    unsigned row[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { row[i] = row_a[i] + cur; opaque(row[i]); }
    stw = stw_a + cur; str = str_a + cur;
    opaque(stw); opaque(str);
    floatx16 Sa[KT];
    bf16x8 ring[RING], Pf[KT][2];
    float mx = -INFINITY, l = 0.f;
    auto rd = [&](int ks) { return lds_read8(row[ks / RSTEP] + (ks % RSTEP) * 32); };
#pragma unroll
    for (int i = 0; i < AH && i < KS; ++i) ring[i] = rd(i);
    fence();
    // S^T = K Q^T: lane <-> row, registers <-> keys
    static_for<KT * KS>([&](auto mc) {
      constexpr int m = decltype(mc)::value, ks = m / KT, kt = m % KT;
      if constexpr (kt == 0 && ks + AH < KS) ring[(ks + AH) % RING] = rd(ks + AH);
      Sa[kt] = mfma32(Kf[kt][ks], ring[ks % RING], ks == 0 ? zero_acc() : Sa[kt]);
      fence();
    });
    const int pv = ui.v0 + min(t * ppt + (n_ >> lg), count - 1), lim = pv < ui.own ? pv : P.B - 1;
    if (!__all(lim >= 32 * KT - 1)) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (32 * kt + 8 * (e >> 2) + 4 * h + (e & 3) > lim) Sa[kt][e] = -INFINITY;
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 16; ++e) mx = fmaxf(mx, Sa[kt][e]);
    mx = halves_max(mx);
    const float mxs = mx * sc;                       // the row maximum in the exponent's units (log2)
    auto exps = [&](int kt, int e) {
      const float p = fast_exp2(__builtin_fmaf(Sa[kt][e], sc, -mxs));
      l += p;
      Pf[kt][e >> 3][e & 7] = (__bf16)p;
    };
#pragma unroll
    for (int e = 0; e < 8; ++e) exps(0, e);
    fence();
    // O^T = V^T P^T, 16 keys at a time, behind its products the next 16 keys' exponentials
    static_for<2 * KT>([&](auto gc) {
      constexpr int g = decltype(gc)::value, kt = g / 2, u2 = g % 2;
      static_for<DT>([&](auto dc) {
        constexpr int dt = decltype(dc)::value, per = 8 / DT;
        Oa[dt] = mfma32(VT[dt][kt][u2], Pf[kt][u2], g == 0 ? zero_acc() : Oa[dt]);
        if constexpr (g + 1 < 2 * KT) static_for<per>([&](auto jc) { constexpr int e = 8 * ((g + 1) % 2) + per * dt + decltype(jc)::value; exps((g + 1) / 2, e); });
        fence();
      });
    });
    l = halves_sum(l);
    inv = 1.0f / l;
    lse = (mxs + fast_log2(l)) * kLn2;
#pragma unroll
    for (int c = 0; c < 4 * DT; ++c) stage(c);
#pragma unroll
    for (int x = 0; x < NT; ++x) read_rows(t & 1, x);
    fence();
#pragma unroll
    for (int x = 0; x < NT; ++x) store_rows(x);
    store_lse(t & 1);
    // ... and the rows of the tile after next in their place
    const Offsets o = offsets(decode(t + 2, raw));
    raw = pair_of(t + 3);
    fence();
    static_for<NT>([&](auto tc) { gather(o, lds0 + cur, tc); });
    fence();
  }
  wait_vm<0>();      // nothing on its way into LDS when the wave ends
}

}  // namespace nsa
