// The backward walk of block-selection attention for 33 .. 64 keys a block and 128 features: one wave per tile, four waves per block.
//
// A tile is 32 rows (32 / G pairs x G heads) against the block's 64 keys.  The walk it takes over from (sel_bwd_dkv_kernel) shares a
// tile between two waves, 32 keys each, with four barriers a tile: of a step's 5200 cycles the matrix cores had 1280, and with all its
// rows in a cache and no stores it took as long as with them (2.69 ms against 2.72 at seq 32k, 32 / 8 heads, 15 blocks + own) - its
// instructions bounded it, not its memory.  Here
//   * a wave keeps the dK and dV of all 64 keys (256 accumulation registers) and walks its own tiles without a barrier; an operand of
//     Q^T or dO^T read from LDS feeds two products.  The four waves of a work-group take every fourth tile of one unit and share the
//     block's K rows in LDS; their sums meet there at the unit's end.
//   * rows come by DMA (buffer_load ... lds), the Q rows of a tile two tiles ahead, its dO rows one, with waits that count what was
//     issued behind them.  Nothing else in the loop waits for memory.
//   * the step is laid out by hand: 80 MFMAs in five runs (S, dP, dV, dK, dQ), behind each of them a share of everything else - the
//     dQ rows of the tile before go out during S, the exponentials run beside dP and dV, the row gathers beside dP and dQ.  The
//     fences keep the compiler to it; up to six plain instructions are free behind an MFMA (32 cycles).
//   * tiles in LDS: groups of four rows, 1 KB each as one DMA instruction writes them, 16 bytes between groups, chunk c of row r at
//     c ^ 4 (r % 4): row reads and transpose loads both without bank conflicts.
//   * work-groups stay and take units by number (an atomic counter; what a unit computes does not depend on who takes it), so that
//     the next unit's lists, K and V rows and first tiles are under way while the sums of the last one are written.
// Measured (MI355X): 2.54 -> 1.86 ms at seq 32k, 32 / 8 heads; 384 -> 269 us with its reduction at seq 4k.  In the loop the gathers
// and stores now run at what the memory gives their pattern (8.3 TB/s); 15 % of the time are the units' ends.  The same walk at 64
// features, where a step has half the MFMAs and the same softmax, was slower than the two-wave walk (190 against 170 us at seq 8k).
#pragma once
#include "nsa_pipe.hpp"
#include "nsa_select_plan.hpp"

namespace nsa {

struct BlockArgs {
  SelPlan P;
  SmallDiv by_sp;
  const __bf16 *q, *k, *v, *dout;
  const float *lse, *delta;
  const char* iws;
  char* bws;
  unsigned* ticket;
  __bf16 *dk, *dv;
};
typedef const BlockArgs __attribute__((address_space(4)))* block_args;

// G >= 4: the four rows of a gather instruction are heads of one pair and have one scalar offset.
// lse, delta: -lse log2 e and -(sum out * d_out - d_lse), as sel_delta_kernel leaves them
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1))) void sel_bwd_block_kernel(const BlockArgs kernel_args) {
  // the arguments are read where they are used: what the loop over the tiles does not need is not worth a register there
  auto args = []() { block_args p = (block_args)__builtin_amdgcn_kernarg_segment_ptr(); asm volatile("" : "+s"(p)); return p; };
  constexpr int D = 128, KS = D / 16, DT = D / 32, NW = 4, KT = 2;
  constexpr int CPR = D / 8, RPI = 64 / CPR, NT = 32 / RPI;                      // 16-byte chunks of a row, rows a DMA instruction, instructions a tile
  constexpr int GB = 1024 + 16, TB = (NT * GB + 255) / 256 * 256, BUFB = 2 * TB; // bytes of a group of rows, of a tile, of a Q and a dO tile
  __shared__ __align__(1024) char tile_s[NW * 2 * BUFB];        // [wave][tile % 2][Q tile | dO tile, then dS^T, then the dQ rows]
  __shared__ __align__(16) char kb_s[2 * TB];                  // the block's K rows
  __shared__ __align__(16) float scal_s[NW][2][64];            // [wave][tile % 2] -lse * log2 e of the tile's rows, then -delta
  __shared__ int ent_s[NW][4][64];                             // [wave][tile % 4] list entry of each row
  __shared__ __align__(8) char* pair_s[NW][4][32];             // [wave][tile % 4] where each row's dQ partial goes
  __shared__ int next_s[2][8];                                 // unit: kv head (-1: none left), index, block, own pairs, list start, range, units of the block
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, n_ = lane & 31, h = lane >> 5;
  const block_args A0 = args();
  const int lg = A0->P.lg, ppt = 32 >> lg, SP = A0->P.SP, S = A0->P.S, blockB = A0->P.B;
  const unsigned per_head = (unsigned)A0->P.n * (unsigned)SP;
  const SmallDiv by_sp = {A0->by_sp.mul, A0->by_sp.sh};
  // byte of 16-byte chunk c of row r in a tile
  auto tile_off = [](int r, int c) { return (r / RPI) * GB + (r % RPI) * (2 * D) + 16 * (c ^ (4 * (r & 3))); };
  typedef __attribute__((address_space(3))) void* lds_p;
  auto lds_addr = [](void* p) { return (unsigned)(unsigned long)(lds_p)p; };
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_addr(tile_s + wave * 2 * BUFB));
  const unsigned scal0 = __builtin_amdgcn_readfirstlane(lds_addr(&scal_s[wave][0][0]));
  const unsigned ent0 = __builtin_amdgcn_readfirstlane(lds_addr(&ent_s[wave][0][0]));
  const unsigned kbase = __builtin_amdgcn_readfirstlane(lds_addr(kb_s));

  // units of kv heads hbase .. hbase + 63, one a lane, as running totals: the next unit's number becomes (kv head, unit) without memory
  int hbase = 0, ubefore = 0, uend = 0;
  auto load_window = [&]() {
    const block_args A = args();
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int hh = hbase + ln;
    int c = hh < A->P.bh ? reinterpret_cast<const int*>(A->iws + A->P.off_unit[2])[(size_t)hh * (A->P.W + 1) + A->P.W] : 0;
    for (int o = 1; o < 64; o <<= 1) { const int x = __shfl_up(c, o, 64); c += ln >= o ? x : 0; }
    uend = ubefore + c;
  };
  // three steps: take a number; find its unit and ask for the record; leave the record in next_s
  unsigned tk = 0;
  int4 rec0 = {0, 0, 0, 0}, rec1 = {0, 0, 0, 0};
  int nbh = -1, nu = 0;
  auto take = [&]() { tk = lane == 0 ? atomicAdd(args()->ticket, 1u) : 0u; };
  auto find = [&]() {
    const int t = __builtin_amdgcn_readfirstlane((int)tk);
    const block_args A = args();
    nbh = -1;
    for (;;) {
      const int total = __builtin_amdgcn_readlane(uend, 63);
      if (t < total) {
        const int l = __popcll(__ballot(uend <= t));
        nbh = hbase + l;
        nu = t - (l ? __builtin_amdgcn_readlane(uend, l - 1) : ubefore);
        break;
      }
      if (hbase + 64 >= A->P.bh) break;
      hbase += 64; ubefore = total;
      load_window();
    }
    if (nbh >= 0) {
      const int4* rec = reinterpret_cast<const int4*>(A->iws + A->P.off_urec[2]) + ((size_t)nbh * A->P.ub[2] + nu) * 2;
      rec0 = rec[0]; rec1 = rec[1];
    }
  };
  auto leave = [&](int slot) {
    if (lane == 0) {
      int* o = next_s[slot];
      o[0] = nbh; o[1] = nu; o[2] = rec0.x; o[3] = rec0.y; o[4] = rec0.z; o[5] = rec0.w; o[6] = rec1.x; o[7] = rec1.y;
    }
  };
  if (wave == 0) { load_window(); take(); find(); leave(0); }

  const int lrow = lane / CPR, pos = lane % CPR;
  const int G = A0->P.g;
  const unsigned sqh = 2u * (unsigned)A0->P.sq[1], sqt = 2u * (unsigned)A0->P.sq[2], soh = 2u * (unsigned)A0->P.so[1], sot = 2u * (unsigned)A0->P.so[2];
  const unsigned chunk0 = 16u * (pos ^ (4 * (lrow & 3)));
  const unsigned vq0 = chunk0 + (unsigned)lrow * sqh, vg0 = chunk0 + (unsigned)lrow * soh;
  const unsigned head_q = (unsigned)(n_ & (G - 1)) * sqh, head_g = (unsigned)(n_ & (G - 1)) * soh;
  const unsigned pair_bytes = (unsigned)G * (D * 2);
  const float scale = A0->P.scale, sc = scale * kLog2e;
  const unsigned head_d = (unsigned)(n_ & (G - 1)) * (D * 2);
  char* const dqpart = A0->bws + A0->P.off_dqpart;
  char* const spare = dqpart + (unsigned long)((unsigned)A0->P.bh * per_head) * pair_bytes;

  // LDS byte addresses of this lane, all of the buffer in use
  constexpr int NR = KS / 2;
  unsigned row_a[NR], krow_a[NR], tr_a[DT], ktr_a[DT], dsr_a, dsw_a, stw_a, str_a, scal_a;
  {
    const int ll = lane & 15, e = ll >> 2, qq = ll & 3, mh = (lane >> 4) & 1;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const unsigned o = tile_off(n_, 4 * i + h);
      row_a[i] = lds0 + o; krow_a[i] = kbase + o;
    }
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      const unsigned o = tile_off(4 * h + e, 4 * i + 2 * mh + (qq >> 1)) + 8 * (qq & 1);
      tr_a[i] = lds0 + o; ktr_a[i] = kbase + o;
    }
    // dS^T: 64 bytes a key, 8-byte piece x at x ^ (key / 4 % 8)
    dsr_a = lds0 + TB + 64 * (4 * h + e) + 8 * ((4 * mh + qq) ^ h);
    dsw_a = lds0 + TB + 64 * n_ + 8 * (h ^ ((n_ >> 2) & 7));
    // dQ rows (2 D bytes) of the tile before: 16-byte chunk c at c ^ (n_ % CPR)
    stw_a = lds0 + BUFB + TB + 2 * D * n_ + 16 * (n_ & (CPR - 1)) + 8 * h;
    str_a = lds0 + BUFB + TB + 2 * D * lrow + 16 * (pos ^ (lrow & (CPR - 1)));
    scal_a = scal0 + 16 * h;
#pragma unroll
    for (int i = 0; i < NR; ++i) { opaque(row_a[i]); opaque(krow_a[i]); }
#pragma unroll
    for (int i = 0; i < DT; ++i) { opaque(tr_a[i]); opaque(ktr_a[i]); }
    opaque(dsr_a); opaque(dsw_a); opaque(stw_a); opaque(str_a); opaque(scal_a);
  }
  int buf = 0, flip = BUFB;             // the tile's buffer, bytes from it to the other one
  auto turn = [&]() {                   // on to the other buffer; the staging addresses follow a tile behind
#pragma unroll
    for (int i = 0; i < NR; ++i) row_a[i] += flip;
#pragma unroll
    for (int i = 0; i < DT; ++i) tr_a[i] += flip;
    dsr_a += flip; dsw_a += flip;
    stw_a -= flip; str_a -= flip;
    scal_a += buf ? -256 : 256;
    flip = -flip;
    buf ^= 1;
  };

  int bh = 0, unit = 0, of_block = 0, blk = 0, own = 0, lst0 = 0, v0 = 0, v1 = 0;
  auto read_next = [&](int slot) {
    const int* o = next_s[slot];
    bh = __builtin_amdgcn_readfirstlane(o[0]); unit = __builtin_amdgcn_readfirstlane(o[1]); blk = __builtin_amdgcn_readfirstlane(o[2]);
    own = __builtin_amdgcn_readfirstlane(o[3]); lst0 = __builtin_amdgcn_readfirstlane(o[4]); v0 = __builtin_amdgcn_readfirstlane(o[5]);
    v1 = __builtin_amdgcn_readfirstlane(o[6]); of_block = __builtin_amdgcn_readfirstlane(o[7]);
  };
  int q_lo = 0, q_hi = 0, q_n = 0, g_lo = 0, g_hi = 0, g_n = 0;      // buffer descriptors of the kv head's Q and dO rows; q_n, g_n = 0: loads touch nothing
  auto desc = [](int lo, int hi, int cnt) {
    rsrc4 r;
    r[0] = __builtin_amdgcn_readfirstlane(lo); r[1] = __builtin_amdgcn_readfirstlane(hi); r[2] = __builtin_amdgcn_readfirstlane(cnt); r[3] = 0x00020000;
    return r;
  };
  const char* scal_base = nullptr;
  int l_lo = 0, l_hi = 0, l_n = 0;        // ... of the unit's list entries
  char* dq_head = nullptr;               // the kv head's dQ partials
  bf16x8 Vf[KT][KS];
  bf16x8 Kraw[64 * CPR / 256];
  // a unit's tensors: descriptors, V operands, this thread's share of the K rows
  int td = threadIdx.x;                 // passed through an empty statement a unit, like the arguments
  auto open_list = [&]() {
    const block_args A = args();
    const unsigned long la = (unsigned long)(reinterpret_cast<const int*>(A->iws + A->P.off_list) + (size_t)bh * A->P.list_cap + lst0), left = 4ul * (unsigned long)(A->P.list_cap - lst0);
    l_lo = (int)(unsigned)la; l_hi = (int)(unsigned)(la >> 32); l_n = left > 0xffffffffu ? -1 : (int)(unsigned)left;
    dq_head = dqpart + (unsigned long)((unsigned)bh * per_head) * pair_bytes;
  };
  auto open_unit = [&]() {
    const block_args A = args();
    asm volatile("" : "+v"(td));
    const int ln = td & 63;
    const int b = bh / A->P.hkv, hk = bh % A->P.hkv;
    const unsigned long qa = (unsigned long)(A->q + b * A->P.sq[0] + (long)(hk * G) * A->P.sq[1]), ga = (unsigned long)(A->dout + b * A->P.so[0] + (long)(hk * G) * A->P.so[1]);
    q_lo = (int)(unsigned)qa; q_hi = (int)(unsigned)(qa >> 32); g_lo = (int)(unsigned)ga; g_hi = (int)(unsigned)(ga >> 32);
    scal_base = reinterpret_cast<const char*>((ln >> 5 ? A->delta : A->lse) + ((size_t)bh * G + (ln & (G - 1))) * A->P.n);
    const unsigned long ka = (unsigned long)(A->k + b * A->P.sk[0] + hk * A->P.sk[1] + (long)blk * blockB * A->P.sk[2]);
    const unsigned long va = (unsigned long)(A->v + b * A->P.sv[0] + hk * A->P.sv[1] + (long)blk * blockB * A->P.sv[2]);
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc((void*)ka, 0, 0x7fffffff, 0x00020000), vr = __builtin_amdgcn_make_buffer_rsrc((void*)va, 0, 0x7fffffff, 0x00020000);
    const unsigned sk = 2u * (unsigned)A->P.sk[2], sv = 2u * (unsigned)A->P.sv[2];
    const int left = A->P.n - blk * blockB, keys = left < blockB ? left : blockB;      // rows behind them are asked for out of range and come as zeros
#pragma unroll
    for (int i = 0; i < 64 * CPR / 256; ++i) {
      const int e = td + 256 * i, row = e / CPR, c = e % CPR;
      Kraw[i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(kr, row < keys ? (int)(row * sk + 16 * c) : (int)0x80000000, 0, 0));
    }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const int kl = 32 * kt + (ln & 31);
      const unsigned o = kl * sv + 16 * (ln >> 5);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) Vf[kt][ks] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(vr, (int)(kl < keys ? o : 0x80000000u) + 32 * ks, 0, 0));
    }
  };
  auto put_k = [&]() {
#pragma unroll
    for (int i = 0; i < 64 * CPR / 256; ++i) {
      const int e = td + 256 * i;
      *reinterpret_cast<bf16x8*>(kb_s + tile_off(e / CPR, e % CPR)) = Kraw[i];
    }
  };
  // DMA of the list entries of the tile at vt_, into ring slot `slot`
  auto dma_entries = [&](int vt_, int slot) {
    const unsigned o = 4u * (unsigned)max(min(vt_ + (n_ >> lg), v1 - 1) - own, 0);
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 3\n\tbuffer_load_dword %2, %3, 0 offen lds" :: "s"(ent0), "s"(slot * 256), "v"(o), "s"(desc(l_lo, l_hi, l_n)) : "memory", "m0", "scc");
  };
  auto entry = [&](int slot) { return *(lds_i)(ent0 + slot * 256 + 4 * lane); };
  // query of this lane's row of the tile at vt_ (its entries have arrived); leaves the pairs' partial rows in pair_s
  auto decode = [&](int vt_, int slot, int raw) {
    const int pv = min(vt_ + (n_ >> lg), v1 - 1);
    const unsigned qd = __umulhi(2u * (unsigned)raw, by_sp.mul) >> by_sp.sh;
    const bool mine = pv < own;
    const int qi = mine ? blk * blockB + pv : (int)qd;
    const unsigned full = mine ? (unsigned)(blk * blockB + pv) * SP + S : (unsigned)raw;
    const bool live = vt_ + (n_ >> lg) < v1;
    pair_s[wave][slot][n_] = (live ? dq_head : spare) + ((unsigned long)(live ? full : 0u) * pair_bytes + head_d);
    return qi;
  };
  // byte offsets of a tile's rows, one scalar a gather instruction.  A scalar that a vector instruction wrote may be an address five wait
  // states later: these are made in a slot of their own, and the first instruction of a run waits itself.
  struct Offsets { int row[NT]; };
  auto offsets = [&](unsigned o) {
    Offsets r;
#pragma unroll
    for (int t = 0; t < NT; ++t) r.row[t] = __builtin_amdgcn_readlane(o, t * RPI);
    return r;
  };
  auto dma_rows = [&](const Offsets& o, unsigned at, unsigned dst, rsrc4 rows, auto tc) {
    constexpr int t = decltype(tc)::value;
    if constexpr (t > 0)
      asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(dst), "v"(at), "s"(rows), "s"(o.row[t]), "n"(t * GB) : "memory", "m0", "scc");
    else
      asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(dst), "v"(at), "s"(rows), "s"(o.row[t]), "n"(t * GB) : "memory", "m0", "scc");
  };
  auto dma_q = [&](const Offsets& o, unsigned bf0, auto tc) { dma_rows(o, vq0, bf0, desc(q_lo, q_hi, q_n), tc); };
  auto dma_g = [&](const Offsets& o, unsigned bf0, auto tc) { dma_rows(o, vg0, bf0 + TB, desc(g_lo, g_hi, g_n), tc); };
  auto dma_scal = [&](int qi, unsigned bf) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" :: "s"(scal0 + bf * 256), "v"(scal_base + 4l * qi) : "memory", "m0");
  };

  floatx16 dKa[DT][KT], dVa[DT][KT], Qa[DT];
  int lrow_ = lrow, lg_ = lg;      // passed through empty statements in the loop: what is derived from them is not worth a register each
  auto stage_dq = [&](int c) {
    const int dt = c / 4, a = c % 4;
    bf16x4 r;
#pragma unroll
    for (int bb = 0; bb < 4; ++bb) r[bb] = (__bf16)(Qa[dt][4 * a + bb] * scale);
    *(lds_x4)(stw_a ^ (unsigned)(16 * c)) = r;
  };
  bf16x8 vv[NT];
  char* pr[NT];
  auto read_dq = [&](int slot, int t) {
    vv[t] = lds_read8((str_a ^ (unsigned)(64 * (t & 3))) + t * 1024);
    pr[t] = pair_s[wave][slot][t * RPI + lrow_];
  };
  auto store_dq = [&](int t) { __builtin_nontemporal_store(vv[t], (glb_x8)(pr[t] + 16 * pos)); };

  constexpr int AH = 4, RING = AH + DT + 1;      // operands read ahead
  constexpr int mB = 2 * KS, mC = 4 * KS, mD = mC + 4 * DT, mE = mD + 4 * DT, mN = mE + 4 * DT;      // first MFMA of each phase
  constexpr int rB = 3 * KS, rC = 4 * KS, rD = rC + 2 * DT, rE = rD + 2 * DT, rN = rE + 4 * (DT + 1);     // first operand of each phase

  __syncthreads();
  int slot = 0;                    // of next_s
  read_next(0);
  if (bh < 0) return;
  int qi1 = 0;                     // query of this lane's row, next tile
  open_list();
#pragma unroll
  for (int i = 0; i < 3; ++i) dma_entries(v0 + (wave + i * NW) * ppt, i);
  open_unit();
  // rows and scalars of a unit's tile i, i = 0, 1 (no dO rows of the second: the loop's first step asks for them)
  auto ask = [&](int i) {
    const int vn = v0 + (wave + i * NW) * ppt;
    qi1 = decode(vn, i, entry(i));
    q_n = g_n = vn < v1 ? -1 : 0;
    const Offsets oq = offsets((unsigned)qi1 * sqt + head_q), og = offsets((unsigned)qi1 * sot + head_g);
    fence();
    dma_scal(qi1, i);
    static_for<NT>([&](auto tc) { dma_q(oq, lds0 + i * BUFB, tc); });
    if (i == 0) static_for<NT>([&](auto tc) { dma_g(og, lds0 + i * BUFB, tc); });
    fence();
  };
  bool first = true;
  for (;;) {
    const int vt0 = v0 + wave * ppt;
    int vt = vt0;
    if (first) {
      wait_vm<0>();
      ask(0);
      ask(1);
      put_k();
      __syncthreads();
      first = false;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      Qa[dt] = zero_acc();
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) { dKa[dt][kt] = zero_acc(); dVa[dt][kt] = zero_acc(); }
    }
    pair_s[wave][3][n_] = spare + head_d;      // "the tile before" the first
    wait_vm<NT + 1>();              // all but the second tile's Q rows and scalars
    fence();

    int tile = 0;
    for (; vt < v1; vt += NW * ppt, ++tile) {
      // Q rows and scalars of this tile (issued two tiles ago; behind them the stores of a tile, this one's dO rows, the next one's entries, scalars and Q rows)
      wait_vm<3 * NT + 2>();
      vt = __builtin_amdgcn_readfirstlane(vt);
      asm volatile("" : "+v"(lrow_), "+s"(lg_));
      const unsigned cur0 = lds0 + buf * BUFB, other0 = lds0 + (buf ^ 1) * BUFB;
      Offsets og, oq;
      int raw2 = 0;
      g_n = vt + NW * ppt < v1 ? -1 : 0;
      int qi2 = 0;
      // wave 0 finds the work-group's next unit, a step a tile
      if (wave == 0 && tile < 3) {
        if (tile == 0) take();
        else if (tile == 1) find();
        else leave(slot ^ 1);
      }

      floatx16 Sa[KT], Pa[KT], nd;
      floatx4 ls[4];
      bf16x8 Pf[KT][2], Sf[KT][2];
      const bool masked = vt < own || vt + ppt > v1 || blockB < 64;
      bf16x8 ring[RING];
      auto rd = [&](auto ic) -> bf16x8 {
        constexpr int i = decltype(ic)::value;
        constexpr unsigned G2 = TB, S2 = 8 / RPI * GB, H2 = 16 / RPI * GB, K2 = 32 / RPI * GB;      // dO tile; 8, 16, 32 rows on
        if constexpr (i < rB) {
          constexpr int ks = i / 3, w = i % 3;
          if constexpr (w == 0) return lds_read8(row_a[ks / 2] + (ks % 2) * 32);
          else return lds_read8(krow_a[ks / 2] + (ks % 2) * 32 + (w - 1) * K2);
        } else if constexpr (i < rC) return lds_read8(row_a[(i - rB) / 2] + ((i - rB) % 2) * 32 + G2);
        else if constexpr (i < rE) {
          constexpr bool isq = i >= rD;
          constexpr int j = isq ? i - rD : i - rC, rh = j / DT, dt = j % DT;
          return lds_read8_tr(tr_a[dt] + rh * H2 + (isq ? 0 : G2), tr_a[dt] + rh * H2 + (isq ? 0 : G2) + S2);
        } else {
          constexpr int kg = (i - rE) / (DT + 1), w = (i - rE) % (DT + 1);
          if constexpr (w == 0) return lds_read8_tr((dsr_a ^ (32 * (kg & 1))) + kg * 1024, (dsr_a ^ (32 * (kg & 1) + 16)) + kg * 1024 + 512);
          else return lds_read8_tr(ktr_a[w - 1] + kg * H2, ktr_a[w - 1] + kg * H2 + S2);
        }
      };
      // operand that MFMA m needs last, and the one up to which operands are read before it (dS^T only behind its stores)
      auto need = [](int m) constexpr {
        return m < mB ? 3 * (m / 2) + 1 + (m & 1) : m < mC ? rB + (m - mB) / 2 : m < mD ? rC + (m - mC) / 2 : m < mE ? rD + (m - mD) / 2
               : rE + (DT + 1) * ((m - mE) / DT) + 1 + (m - mE) % DT;
      };
      auto upto = [need](int m) constexpr {
        const int x = need(m) + AH;
        return m < mD + DT && x >= rE ? rE - 1 : x < rN ? x : rN - 1;
      };
      auto read_to = [&](auto fromc, auto toc) {
        constexpr int from = decltype(fromc)::value, to = decltype(toc)::value;
        if constexpr (to >= from) static_for<to - from + 1>([&](auto jc) {
          constexpr int i = from + decltype(jc)::value;
          ring[i % RING] = rd(std::integral_constant<int, i>{});
        });
      };
      auto lse4 = [&](int a) { return *(lds_f4)(scal_a + 32 * a); };
      auto exps = [&](int kt, int e) {
        const float p = fast_exp2(__builtin_fmaf(Sa[kt][e], sc, ls[e >> 2][e & 3]));
        Sa[kt][e] = p;
        Pf[kt][e >> 3][e & 7] = (__bf16)p;
      };
      auto dss = [&](int kt, int e) { Sf[kt][e >> 3][e & 7] = (__bf16)(Sa[kt][e] * Pa[kt][e]); };

      read_to(std::integral_constant<int, 0>{}, std::integral_constant<int, upto(0) - 1>{});
      fence();
      static_for<mN>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        constexpr int lo = m == 0 ? upto(0) : upto(m - 1) + 1, hi = upto(m);
        read_to(std::integral_constant<int, lo>{}, std::integral_constant<int, hi>{});
        constexpr int i = need(m);
        if constexpr (m < mB) {
          constexpr int ks = m / 2, kt = m & 1;
          Sa[kt] = mfma32(ring[(3 * ks) % RING], ring[i % RING], ks == 0 ? zero_acc() : Sa[kt]);
          constexpr int per = 4 * DT / KS, rpt = NT / (KS / 2);      // dQ chunks of the tile before, over the first half of this phase
          if constexpr (m < KS) static_for<per>([&](auto jc) { stage_dq(per * m + decltype(jc)::value); });
          else {
            if constexpr (m >= KS + 2 && m < KS + 2 + KS / 2) static_for<rpt>([&](auto jc) { store_dq(rpt * (m - KS - 2) + decltype(jc)::value); });
            if constexpr (m < KS + KS / 2) static_for<rpt>([&](auto jc) { read_dq((tile + 3) & 3, rpt * (m - KS) + decltype(jc)::value); });
          }
          if constexpr (m == mB - 1) og = offsets((unsigned)qi1 * sot + head_g);
          if constexpr (m == mB - 4) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
              const floatx4 d4 = *(lds_f4)(scal_a + 128 + 32 * a);
#pragma unroll
              for (int bb = 0; bb < 4; ++bb) nd[4 * a + bb] = d4[bb];
            }
          }
        } else if constexpr (m < mC) {
          constexpr int ks = (m - mB) / 2, kt = m & 1;
          Pa[kt] = mfma32(ring[i % RING], Vf[kt][ks], ks == 0 ? nd : Pa[kt]);
          constexpr int per = 16 / (2 * KS);             // exponentials of rows 0 .. 15
          if constexpr (m == mB) { ls[0] = lse4(0); ls[1] = lse4(1); }
          if constexpr (m == mC - 3) { ls[2] = lse4(2); ls[3] = lse4(3); }
          static_for<per>([&](auto jc) { constexpr int c = per * (m - mB) + decltype(jc)::value; exps(c & 1, c >> 1); });
          if constexpr ((m & 1) && (m - mB) / 2 < NT) dma_g(og, other0, std::integral_constant<int, (m - mB) / 2>{});
        } else if constexpr (m < mD) {
          constexpr int c0 = (m - mC) / 2, rh = c0 / DT, dt = c0 % DT, kt = m & 1;
          mfma32_acc<c0 % DT == 0>(dVa[dt][kt], ring[i % RING], Pf[kt][rh]);
          if constexpr (m - mC < 2 * DT) {               // exponentials of rows 16 .. 31
            constexpr int per = 16 / (2 * DT);
            static_for<per>([&](auto jc) { constexpr int c = per * (m - mC) + decltype(jc)::value; exps(c & 1, 8 + (c >> 1)); });
          } else {
            constexpr int per = 32 / (2 * DT);
            static_for<per>([&](auto jc) { constexpr int c = per * (m - mC - 2 * DT) + decltype(jc)::value; dss(c & 1, c >> 1); });
          }
        } else if constexpr (m < mE) {
          constexpr int c0 = (m - mD) / 2, rh = c0 / DT, dt = c0 % DT, kt = m & 1;
          mfma32_acc<c0 % DT == 0>(dKa[dt][kt], ring[i % RING], Sf[kt][rh]);
          constexpr int per = 8 / DT;
          if constexpr (m - mD < DT) static_for<per>([&](auto jc) {      // dS^T over the dO tile, which nothing reads any more
            constexpr int c = per * (m - mD) + decltype(jc)::value, k2 = c & 1, a = c >> 1;
            bf16x4 t4;
#pragma unroll
            for (int bb = 0; bb < 4; ++bb) t4[bb] = Sf[k2][a >> 1][4 * (a & 1) + bb];
            *(lds_x4)((dsw_a ^ (unsigned)(16 * a)) + k2 * 2048) = t4;
          });
          if constexpr (m == mD) { wait_vm<3 * NT + 1>(); raw2 = entry((tile + 2) & 3); }      // (entries: issued a tile ago, with three runs of rows behind them)
          if constexpr (m == mE - 3) qi2 = decode(vt + 2 * NW * ppt, (tile + 2) & 3, raw2);
          if constexpr (m == mE - 1) { oq = offsets((unsigned)qi2 * sqt + head_q); q_n = vt + 2 * NW * ppt < v1 ? -1 : 0; }
        } else {
          constexpr int g0 = (m - mE) / DT, dt = (m - mE) % DT;
          Qa[dt] = mfma32(ring[i % RING], ring[(rE + (DT + 1) * g0) % RING], g0 == 0 ? zero_acc() : Qa[dt]);
          if constexpr (m == mE) { dma_entries(vt + 3 * NW * ppt, (tile + 3) & 3); dma_scal(qi2, buf); }
          constexpr int every = 4 * DT / NT;
          if constexpr ((m - mE) % every == every - 1) dma_q(oq, cur0, std::integral_constant<int, (m - mE) / every>{});
        }
        fence();
        if constexpr (m == mB - 1) {
          if (masked) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int pv = vt + ((8 * (e >> 2) + 4 * h + (e & 3)) >> lg_);
              const int lim = pv >= v1 ? -1 : pv < own ? pv : blockB - 1;
#pragma unroll
              for (int kt = 0; kt < KT; ++kt)
                if (32 * kt + n_ > lim) Sa[kt][e] = -INFINITY;
              fence();
            }
          }
          fence();
        }
        if constexpr (m + 1 < mN && upto(m + 1) >= rB && upto(m) < rB) {      // this tile's dO rows: issued a tile ago
          constexpr int done = m + 1 - KS - 2, stores = done > KS / 2 ? NT : done > 0 ? done * (NT / (KS / 2)) : 0;
          wait_vm<NT + 2 + stores>();
          fence();
        }
      });
      qi1 = qi2;
      turn();
    }
    if (wave == 0 && tile < 3) {      // the steps that the tiles left out
      if (tile == 0) take();
      if (tile <= 1) find();
      leave(slot ^ 1);
    }
    if (tile > 0) {      // the last tile's rows
#pragma unroll
      for (int c = 0; c < 4 * DT; ++c) stage_dq(c);
#pragma unroll
      for (int t = 0; t < NT; ++t) read_dq((tile + 3) & 3, t);
      fence();
#pragma unroll
      for (int t = 0; t < NT; ++t) store_dq(t);
    }
    fence();
    if (tile > 0) wait_vm<NT>();      // nothing is on its way into LDS any more
    else wait_vm<0>();
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // ... and the last MFMAs have written their results
    fence();
    if (buf) turn();
    const int done_bh = bh, done_unit = unit, done_blk = blk;
    const bool single_unit = of_block == 1;
    __syncthreads();
    slot ^= 1;
    read_next(slot);
    const bool more = bh >= 0;
    if (more) {
      open_list();
#pragma unroll
      for (int i = 0; i < 3; ++i) dma_entries(v0 + (wave + i * NW) * ppt, i);
      open_unit();
    }
    const block_args A = args();
    asm volatile("" : "+v"(td));
    const int ln = td & 63;
    // the four waves' sums, half a tensor at a time through their second buffers: float4 chunk c of key row kl at c ^ (kl % chunks)
    constexpr int FPR = D / 8;             // float4 chunks per key and half
    const int keys = min(blockB, A->P.n - done_blk * blockB);
    float* part = reinterpret_cast<float*>(A->bws + A->P.off_dkvpart) + ((size_t)done_bh * A->P.ub_kv + done_unit) * (2 * 32 * KT * D);
#pragma unroll
    for (int round = 0; round < 4; ++round) {
      const int which = round >> 1, half = round & 1;
#pragma unroll
      for (int d2 = 0; d2 < DT / 2; ++d2)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            const int dt = half * (DT / 2) + d2;
            floatx4 x;
#pragma unroll
            for (int bb = 0; bb < 4; ++bb) x[bb] = which == 0 ? dKa[dt][kt][4 * a + bb] : dVa[dt][kt][4 * a + bb];
            const int kl = 32 * kt + (ln & 31), c = 8 * d2 + 2 * a + (ln >> 5);
            *reinterpret_cast<floatx4*>(tile_s + (wave * 2 + 1) * BUFB + 16 * (kl * FPR + (c ^ (kl & (FPR - 1))))) = x;
          }
      __syncthreads();
      floatx4 sum[64 * FPR / 256];
#pragma unroll
      for (int i = 0; i < 64 * FPR / 256; ++i) {
        const int e = td + 256 * i, kl = e / FPR, c = e % FPR, p = 16 * (kl * FPR + (c ^ (kl & (FPR - 1))));
        sum[i] = *reinterpret_cast<const floatx4*>(tile_s + BUFB + p);
#pragma unroll
        for (int w = 1; w < NW; ++w) sum[i] += *reinterpret_cast<const floatx4*>(tile_s + (2 * w + 1) * BUFB + p);
      }
      __syncthreads();
      if (round == 0 && more) {      // the next unit's first tile, into the first buffers
        wait_vm<0>();
        ask(0);
        put_k();
      }
      if (round == 3 && more) {      // ... and its second tile's Q rows
        ask(1);
      }
#pragma unroll
      for (int i = 0; i < 64 * FPR / 256; ++i) {
        const int e = td + 256 * i, kl = e / FPR, c = e % FPR, col = half * (D / 2) + 4 * c;
        if (single_unit) {
          const float mlt = which == 0 ? scale : 1.0f;
          if (kl < keys) store4_bf16((which == 0 ? A->dk : A->dv) + ((size_t)done_bh * A->P.n + (size_t)done_blk * blockB + kl) * D + col, sum[i][0] * mlt, sum[i][1] * mlt, sum[i][2] * mlt, sum[i][3] * mlt);
        } else {
          *reinterpret_cast<floatx4*>(part + which * 64 * D + (size_t)kl * D + col) = sum[i];
        }
      }
    }
    if (!more) break;
  }
}

}  // namespace nsa
