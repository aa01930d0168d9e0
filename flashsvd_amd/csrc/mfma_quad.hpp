// Projections and head expansions of prompts: the kernel (rules and launches: mfma_quad.hip and mfma_quad_heads.hip).
//
// A workgroup is four waves, one per SIMD, that own a quarter of the output tile each: (16 TM) x (16 TN) of (32 TM) x (32 TN).  What
// bounds these products beside the matrix cores is the way of the operands into the registers: the loads of a walk reach LDS at 50 to 90 bytes
// per ns and compute unit, products and reads taken out (512 x 3072 x 4096 18.6 of 20.0 us, 8192 x 8192 x 8192 490 of 717), and a fragment read by
// every wave that shares it costs LDS cycles and, under the chip's power limit, clock.  Four waves of 128 x 128 read two thirds of what eight of 128 x
// 64 do for the same products: 8192 x 8192 x 8192 723 us (1.52 PFLOP/s; eight waves 1.31 PFLOP/s at 16384 x 4992 x 4096, this 1.43; products
// alone, operands fixed, 1.65 to 1.7 at the clock that the chip then keeps).
//
// One wave per SIMD has nobody to fill its gaps, so the order is laid down by hand: a K step of 64 is two slices of 32, a slice's
// products run while the fragments of the next one are read into the other register set, one read every RD products, and loads for a
// later step go out between the products as well, one every LD (all at once, in front of the products, stalls the wave at the
// issue: 783 against 718 us).  One barrier per step, in its middle: behind it every wave has read the step to its end and its share of
// the next one has landed.  W rows may run one step further ahead of the products than x rows (NSW = NSX + 1; a weight comes from HBM, and
// 160 KB hold no third stage of a 256 x 256 tile): their loads then fill the first slice, those of x the second (487 -> 469 us).
// Accumulators of the forms with one workgroup per compute unit are written as AGPR operands of the product: left to the compiler
// they are moved between both halves of the register file in every step (1043 against 720 us).
//
// The walk over tiles is one stream: load cursors run ahead of the products across tiles, so the first stages of the next tile land
// while a finished tile leaves the registers.  Loads past a workgroup's last step have no record in range and move nothing; the
// step count needs no second walk for its end.
//
// LDS rows are 128 bytes (64 of K), their eight 16-byte pieces XOR-swizzled by row % 8 as in mfma_gemm.hip.  RAG: K that is no multiple of
// 64 and rows on the 4-byte grid; the thread that loaded a piece past the end of its row clears what lies past it in LDS before
// the step's barrier.
#pragma once
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "quad_costs.hpp"

namespace fsvd {

enum QuadEpi { kQuadPlain = 0, kQuadPair = 1, kQuadHeads = 2, kQuadShare = 3 };
constexpr int kQuadThreads = 256, kQuadRow = 128;

struct QuadArgs {
  MfmaArgs a[3];                                     // heads: up to three expansions of the same token rows
  ExpandEpi ep[3];
  int first[4];                                      // heads: column tiles of problem i are [first[i], first[i + 1])
  int nt, mt;                                        // column and row tiles
  float us;                                          // what the launch is expected to take
  AheadList next;                                    // what workgroups without a tile ask for
  int shares, per; float* part;                      // kQuadShare: workgroups per tile, K steps of each (the last may have fewer), their sums; CUT: per
};

// two tiles' words of a row of 16 lanes become consecutive words (see mfma_big.hip)
__device__ __forceinline__ void quad_swap_rows(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// four elements at any element's address
typedef uint32_t u32x2_any_t __attribute__((ext_vector_type(2), aligned(2)));

constexpr bool quad_asks(int tm, int tn) { return tm * tn < 32; }      // the tiles of many rows are left out
static int quad_ahead(QuadArgs& q, int64_t wgs, int64_t rows) {
  const AheadChoice c = ahead_choice(q.a[0].next, q.us, q.a[0].B, rows, compute_units() - wgs);
  q.next = c.ranges;
  return c.workgroups;
}

constexpr bool quad_stream(int tm, int tn) { return tm * tn >= 24; }

// H = 2: the first 64 of every 128 of K and the second 64 are added up apart and then together; CUT: K in ranges of args.per steps, their sums
// added in order (the order of the sums in which the rows of these shapes were added before: the same bits).
template <int DT, int EPI, int TM, int TN, int NSX, int NSW, int OCC, bool RAG, int H, bool CUT>
__global__ __launch_bounds__(kQuadThreads, OCC) void gemm_quad_kernel(QuadArgs args) {
  typedef E16<DT> E;
  typedef typename E::frag_t frag_t;
  constexpr bool PAIR = EPI == kQuadPair, HEADS = EPI == kQuadHeads, SHARE = EPI == kQuadShare;
  constexpr bool AGPR = OCC == 1;
  constexpr int BM = 32 * TM, BN = 32 * TN, LX = BM / 32, LW = BN / 32, NF = TM + TN, NM = TM * TN;
  // several tiles per workgroup as one stream of steps; small tiles leave that to the launch (their steps are as short as the cursors' upkeep)
  constexpr bool STREAM = quad_stream(TM, TN);
  constexpr bool WAHEAD = NSW > NSX;                 // W loads in the first slice of a step, else all behind its middle
  static_assert(NSX >= 2 && (NSW == NSX || NSW == NSX + 1), "stages");
  static_assert(!HEADS || TN % 2 == 0, "rotation pairs in one wave");
  static_assert(!RAG || !SHARE, "shares take whole steps");
  static_assert((H == 1 && !CUT) || (EPI == kQuadPlain && !RAG && !(H == 2 && CUT)), "orders of the sums: single matrices of whole steps");
  constexpr int kSX = BM * kQuadRow, kSW = BN * kQuadRow, kW0 = NSX * kSX;
  constexpr int RD = NM >= 3 * NF ? (NM >= 64 ? 4 : 2) : (NM >= 2 * NF ? 2 : 1);
  constexpr int kLoads = WAHEAD ? (LX > LW ? LX : LW) : LX + LW, LD = NM / kLoads > 0 ? NM / kLoads : 1;
  extern __shared__ __align__(16) unsigned char quad_smem[];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int wm = __builtin_amdgcn_readfirstlane(wave >> 1), wn = __builtin_amdgcn_readfirstlane(wave & 1);

  // Every XCD takes one contiguous run of tiles in bands of eight row tiles walked column by column, its workgroups neighbouring
  // tiles of it at a time, so that they share their x and W rows in one L2 (shares: a K range of all tiles before the next range).
  const int NT = args.nt, MT = args.mt, tiles = NT * MT, all = SHARE ? tiles * args.shares : tiles;
  const int xcd = blockIdx.x & 7, quota = all >> 3, rem = all & 7;
  const int run0 = xcd * quota + min(xcd, rem), run_n = quota + (xcd < rem ? 1 : 0);
  const int wgs = ((int)gridDim.x - xcd + 7) >> 3;   // workgroups of this XCD
  struct Where { int pi, m0, n0, t, share, k0, steps; };
  const auto where = [&](int i) {
    Where w;
    w.share = SHARE ? (run0 + i) / tiles : 0;
    w.t = run0 + i - w.share * tiles;
    const int band = w.t / (8 * NT), tb = w.t - band * 8 * NT, bh = min(8, MT - band * 8), col = tb / bh;
    w.pi = !HEADS ? 0 : (col >= args.first[2] ? 2 : (col >= args.first[1] ? 1 : 0));
    w.m0 = (band * 8 + tb - col * bh) * BM;
    w.n0 = (col - args.first[w.pi]) * BN;
    const int ksteps = (args.a[w.pi].K + 63) >> 6;
    w.k0 = SHARE ? w.share * args.per : 0;
    w.steps = SHARE ? min(args.per, ksteps - w.k0) : (PAIR ? 2 : 1) * ksteps;
    return w;
  };
  int ti = blockIdx.x >> 3;
  if (ti >= run_n) {
    if constexpr (quad_asks(TM, TN)) {
#pragma unroll
      for (int i = 0; i < 3; ++i) request_ahead<kQuadThreads>(args.next.r[i], blockIdx.x - all, gridDim.x - all, tid);
    }
    return;
  }

  // ---- load cursors.  Eight threads per row, rows tid / 8 + 32 j of each operand: a lane's byte offset holds its row and piece, the
  // base address the K step.  Offsets fit 32 bits (the launcher checks), rows past the end are clamped to the last one.
  const int lrow = tid >> 3, lpiece = ((tid & 7) ^ (lrow & 7)) * 16;
  struct Cursor { int ti, s, steps; const uint16_t* p; uint32_t bytes; const uint16_t* p2; uint32_t bytes2; int records; };
  // bytes: from p to the end of the operand; records: what the next step may read (ragged rows end where the operand ends; otherwise
  // nothing past it is asked for), none behind a workgroup's last step
  const auto set_records = [](Cursor& c) {
    int live;                                        // all ones in front of the last step's end (written out: a select would cross the vector unit)
    asm("s_cmp_lt_i32 %1, %2\n\ts_cselect_b32 %0, -1, 0" : "=s"(live) : "s"(c.s), "s"(c.steps) : "scc");
    c.records = RAG ? (int)c.bytes & live : live;
  };
  Cursor cx, cw;
  uint32_t xo[LX], wo[LW];
  const auto aim_x = [&](const Where& w) {
    const MfmaArgs& a = args.a[w.pi];
    const ExpandEpi& ep = args.ep[w.pi];
    cx.s = 0;
    cx.steps = w.steps;
    cx.p = a.x + w.k0 * 64;
    const int64_t top = HEADS ? (int64_t)((a.B - 1) / ep.M) * ep.sp_b + (int64_t)(ep.M - 1) * ep.sp_m : (int64_t)(a.B - 1) * a.ldx;
    cx.bytes = (uint32_t)((top + a.K - w.k0 * 64) * 2 + 2) & ~3u;
    if (PAIR) { cx.p2 = a.x + a.up_off; cx.bytes2 = cx.bytes; }
#pragma unroll
    for (int j = 0; j < LX; ++j) {
      const int r = min(w.m0 + lrow + 32 * j, a.B - 1);
      if (HEADS) {
        const int b = r / ep.M;
        xo[j] = (uint32_t)((b * ep.sp_b + (r - b * ep.M) * ep.sp_m) * 2) + lpiece;
      } else {
        xo[j] = (uint32_t)(r * a.ldx * 2) + lpiece;
      }
    }
  };
  const auto aim_w = [&](const Where& w) {
    const MfmaArgs& a = args.a[w.pi];
    cw.s = 0;
    cw.steps = w.steps;
    cw.p = a.W + w.k0 * 64;
    cw.bytes = (uint32_t)(((int64_t)(a.N - 1) * a.ldw + a.K - w.k0 * 64) * 2 + 2) & ~3u;
    if (PAIR) { cw.p2 = a.W2; cw.bytes2 = cw.bytes; }
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      const int c = lrow + 32 * j;
      int r;
      if (HEADS) {                                   // sixteen columns of a head and the sixteen 64 past them in turn
        const int unit = w.n0 / 32 + (c >> 5);
        r = (unit >> 2) * 128 + ((c >> 4) & 1) * 64 + (unit & 3) * 16 + (c & 15);
      } else {
        r = w.n0 + c;
      }
      wo[j] = (uint32_t)(min(r, a.N - 1) * a.ldw * 2) + lpiece;
    }
  };
  const auto step_on = [&](Cursor& c, auto aim) {
    ++c.s;
    c.p += 64;
    if (RAG) c.bytes -= 128;
    if (PAIR && c.s * 2 == c.steps) {
      c.p = c.p2;
      if (RAG) c.bytes = c.bytes2;
    }
    if (STREAM && c.s == c.steps) {
      c.ti += wgs;
      if (c.ti < run_n) aim(where(c.ti));                // else the step count stays at its end: nothing is in range any more
    }
    set_records(c);
  };
  const uint32_t my = (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 1024;
  const auto load_x = [&](int stage, int q) {
#if defined(__HIP_DEVICE_COMPILE__)
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(cx.p), 0, cx.records, 0x00020000u);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(quad_smem + stage * kSX + my + q * 32 * kQuadRow), 16, (int)xo[q], 0, 0, 0);
#endif
  };
  const auto load_w = [&](int stage, int q) {
#if defined(__HIP_DEVICE_COMPILE__)
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(cw.p), 0, cw.records, 0x00020000u);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(quad_smem + kW0 + stage * kSW + my + q * 32 * kQuadRow), 16, (int)wo[q], 0, 0, 0);
#endif
  };
  const auto barrier = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // ragged: what this thread loaded past the end of its rows, cleared in the stages of the step that holds the end
  const auto clear_tail = [&](int K, int sx, int sw) {
    asm volatile("" ::: "memory");
    const int left = K - ((K - 1) & ~63) - lpiece / 2;          // elements of the row from this thread's piece on
    if (left < 8) {
      const auto fix = [&](unsigned char* p) {
        u32x4_t v = *reinterpret_cast<const u32x4_t*>(p);
        uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = left >= 2 * e + 2 ? w[e] : (left == 2 * e + 1 ? w[e] & 0xffffu : 0u);
        *reinterpret_cast<u32x4_t*>(p) = u32x4_t{w[0], w[1], w[2], w[3]};
      };
#pragma unroll
      for (int q = 0; q < LX; ++q) fix(quad_smem + sx * kSX + q * 32 * kQuadRow + tid * 16);
#pragma unroll
      for (int q = 0; q < LW; ++q) fix(quad_smem + kW0 + sw * kSW + q * 32 * kQuadRow + tid * 16);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
  };

  // ---- fragments and products
  const uint32_t fxo = (wm * 16 * TM + lr) * kQuadRow, fwo = kW0 + (wn * 16 * TN + lr) * kQuadRow;
  struct Frags { frag_t x[TM], w[TN]; };
  Frags f0, f1;
  f32x4_t accs[H][TM][TN];
  auto& acc = accs[0];
  const auto clear = [&] {
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) accs[h][i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // two wait states between these writes and a product that adds to them, which the compiler does not see
    if constexpr (AGPR) {
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) asm volatile("" : "+a"(accs[h][i][j]));
      asm volatile("s_nop 3");
    }
  };
  const auto read1 = [&](Frags& f, int sx, int sw, int kk, int q) {
    const unsigned char* base = quad_smem + ((kk * 4 + lg) ^ (lr & 7)) * 16;
    if (q < TN) f.w[q < TN ? q : 0] = *reinterpret_cast<const frag_t*>(base + sw * kSW + fwo + q * 16 * kQuadRow);
    else f.x[q >= TN ? q - TN : 0] = *reinterpret_cast<const frag_t*>(base + sx * kSX + fxo + (q - TN) * 16 * kQuadRow);
  };
  // the products of one slice; between(q) in front of product q
  const auto sweep = [&](const Frags& f, f32x4_t (&acc)[TM][TN], auto between) {
#pragma unroll
    for (int q = 0; q < NM; ++q) {
      between(q);
      const int i = q / TN, j = q % TN;
      if constexpr (AGPR) {
        if constexpr (DT == 0) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(f.w[j]), "v"(f.x[i]));
        else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(f.w[j]), "v"(f.x[i]));
      } else {
        acc[i][j] = E::mfma(f.w[j], f.x[i], acc[i][j]);
      }
      if (q % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // W steps requested ahead of the walk; loads in flight behind the first step's, and behind the next step's in the middle of a step
  constexpr int NP = WAHEAD ? NSW - 1 : NSW;
  constexpr int kPre = (NSX - 1) * LX + (NP - 1) * LW, kMid = (NSX - 2) * LX + (NSW - 2) * LW;
  static_assert(kPre < 64 && kMid < 64, "load counter");
  constexpr int kTail = (NM + RD - 1) / RD;          // reads that fit between the products
  int sx = 0, sw = 0;
  // large tiles: a walk's first fragments are read again at its start instead of being kept across the epilogue, which needs the registers
  constexpr bool AGAIN = NM > 36 || (PAIR && NM > 20);
  const auto first_reads = [&] {
#pragma unroll
    for (int q = 0; q < NF; ++q) read1(f0, sx, sw, 0, q);
  };
  const auto walk = [&](const int steps) {
    if constexpr (AGAIN) first_reads();
    const auto step = [&](const int s, f32x4_t (&acc)[TM][TN]) {
      const int pw = sw == 0 ? NSW - 1 : sw - 1;
      sweep(f0, acc, [&](int q) {
        if (q % RD == 0 && q / RD < NF) read1(f1, sx, sw, 1, q / RD);
        if (WAHEAD && q % LD == LD - 1 && q / LD < LW) load_w(pw, q / LD < LW ? q / LD : 0);
      });
#pragma unroll
      for (int q = kTail; q < NF; ++q) read1(f1, sx, sw, 1, q);
      if (WAHEAD) {
#pragma unroll
        for (int q = NM / LD; q < LW; ++q) load_w(pw, q);
        step_on(cw, aim_w);
      }
      const int nx = sx == NSX - 1 ? 0 : sx + 1, nw = sw == NSW - 1 ? 0 : sw + 1;
      // this wave has read the step to its end, and its loads of the next one have landed (younger ones may be under way)
      __builtin_amdgcn_s_waitcnt(0x0070 | (kMid & 15) | ((kMid >> 4) << 14));
      if constexpr (RAG) {
        if (s + 2 == steps) clear_tail(args.a[0].K, nx, nw);       // the next step is the last of its rows (two steps at least)
      }
      barrier();
      sweep(f1, acc, [&](int q) {
        if (q % RD == 0 && q / RD < NF) read1(f0, nx, nw, 0, q / RD);
        if (q % LD == LD - 1) {
          const int l = q / LD;
          if (l < LX) load_x(sx, l < LX ? l : 0);
          else if (!WAHEAD && l < LX + LW) load_w(sw, l >= LX && l < LX + LW ? l - LX : 0);
        }
      });
#pragma unroll
      for (int q = NM / LD; q < LX + (WAHEAD ? 0 : LW); ++q) {
        if (q < LX) load_x(sx, q < LX ? q : 0);
        else load_w(sw, q >= LX ? q - LX : 0);
      }
      step_on(cx, aim_x);
      if (!WAHEAD) step_on(cw, aim_w);
#pragma unroll
      for (int q = kTail; q < NF; ++q) read1(f0, nx, nw, 0, q);
      sx = nx;
      sw = nw;
    };
    for (int s = 0; s < steps; s += H) {
      step(s, accs[0]);
      if constexpr (H == 2) step(s + 1, accs[1]);
    }
  };

  Where cur = where(ti);
  // what the epilogue of small tiles reads, requested ahead of the operands: residual rows, or position and rotation rows of all rows
  constexpr int U = HEADS ? TN / 2 : 1;              // rotation units of a wave
  constexpr bool EARLY = HEADS ? TM * U <= (AGPR ? 16 : 8) : (EPI == kQuadPlain && TN % 2 == 0 && NM <= (AGPR ? 32 : 16));
  // The lane's place in a tile, for the epilogue: a value of its own per tile, so that the addresses which follow from it are not kept in
  // registers through the products.
  struct Lane { int lr, lg, tj, c8; };               // after a swap: this lane's tile of two, its eight columns
  const auto lane_now = [&] {
    int l = lane;
    asm volatile("" : "+v"(l));
    return Lane{l & 15, l >> 4, (l >> 4) & 1, (l >> 5) * 8};
  };
  constexpr int RJ = EPI == kQuadPlain && EARLY ? TN / 2 : 1;
  typedef u32x4_t Res[EPI == kQuadPlain ? TM : 1];
  Res rs[RJ];
  constexpr int G = !HEADS ? 1 : (EARLY ? TM : (TM * U <= 16 ? TM : TM / 2));      // rows whose rotation is held at a time
  struct Rows { int pos[G]; u32x2_t cr[G][U], sr[G][U]; };
  Rows early_rows;
  const auto request = [&](const Lane& L, int jp, Res& into) {  // residual pieces of column pair jp
    const MfmaArgs& a = args.a[0];
    const int n = min(cur.n0 + wn * 16 * TN + (2 * jp + L.tj) * 16 + L.c8, a.N - 8);       // a piece past the row's end is not used
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = min(cur.m0 + wm * 16 * TM + i * 16 + L.lr, a.B - 1);
      into[EPI == kQuadPlain ? i : 0] = *reinterpret_cast<const u32x4_any_t*>(a.res + (int64_t)m * a.ldres + n);
    }
  };
  const auto request_rows = [&](const Lane& L, int i0, Rows& R) {            // positions and rotation rows of row tiles i0 .. i0 + G - 1
    const MfmaArgs& a = args.a[cur.pi];
    const ExpandEpi& ep = args.ep[cur.pi];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int r = min(cur.m0 + wm * 16 * TM + (i0 + g) * 16 + L.lr, a.B - 1), b = r / ep.M;
      R.pos[g] = (ep.positions ? ep.positions[b] : ep.pos0) + r - b * ep.M;
    }
    if (ep.cos) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int64_t row = (int64_t)min(max(R.pos[g], 0), ep.rope_len - 1) * 64;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t at = row + ((cur.n0 / 32 + wn * U + u) & 3) * 16 + L.lg * 4;
          R.cr[g][u] = *reinterpret_cast<const u32x2_any_t*>(ep.cos + at);
          R.sr[g][u] = *reinterpret_cast<const u32x2_any_t*>(ep.sin + at);
        }
      }
    }
  };
  const auto request_early = [&] {
    if constexpr (HEADS && EARLY) request_rows(lane_now(), 0, early_rows);
    if constexpr (EPI == kQuadPlain && EARLY) {
      if (args.a[0].res) {
        const Lane L = lane_now();
#pragma unroll
        for (int jp = 0; jp < TN / 2; ++jp) request(L, jp, rs[jp < RJ ? jp : 0]);
      }
    }
  };
  request_early();

  aim_x(cur);
  aim_w(cur);
  cx.ti = cw.ti = ti;
  set_records(cx);
  set_records(cw);
#pragma unroll
  for (int s = 0; s < (NSX > NP ? NSX : NP); ++s) {
    if (s < NP) {
#pragma unroll
      for (int q = 0; q < LW; ++q) load_w(s, q);
      step_on(cw, aim_w);
    }
    if (s < NSX) {
#pragma unroll
      for (int q = 0; q < LX; ++q) load_x(s, q);
      step_on(cx, aim_x);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0f70 | (kPre & 15) | ((kPre >> 4) << 14));
  barrier();
  if constexpr (!AGAIN) first_reads();

  for (;;) {
    const bool more = STREAM && ti + wgs < run_n;
    uint32_t act[PAIR ? TM : 1][PAIR ? TN : 1][2];   // the pair: silu(gate), rounded, two to a word
    // the last products have left the matrix cores (16 wait states; the compiler does not see them in the product's text)
    const auto settle = [&] {
      if constexpr (AGPR) {
        asm volatile("s_nop 15\n\ts_nop 7" : "+a"(accs[H - 1][TM - 1][TN - 1]));
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) asm volatile("" : "+a"(accs[h][i][j]));
      }
    };
    clear();
    if constexpr (PAIR) {
      walk(cur.steps / 2);
      settle();
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const uint32_t g = E::pack2(acc[i][j][2 * w], acc[i][j][2 * w + 1]);
            act[i][j][w] = E::pack2(silu_f32(E::lo(g)), silu_f32(E::hi(g)));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      clear();
      walk(cur.steps / 2);
    } else if constexpr (CUT) {
      f32x4_t sum[TM][TN];
      for (int s = 0; s < cur.steps; s += args.per) {
        if (s) clear();
        walk(min(args.per, cur.steps - s));
        settle();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) sum[i][j] = s ? sum[i][j] + acc[i][j] : acc[i][j];
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = sum[i][j];
    } else {
      walk(cur.steps);
    }
    settle();
    if constexpr (H == 2) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += accs[1][i][j];
    }

    if constexpr (SHARE) {                           // the sums as they lie in the accumulators, for the launch that adds them
      f32x4_t* mine = reinterpret_cast<f32x4_t*>(args.part) + ((size_t)cur.t * args.shares + cur.share) * NM * kQuadThreads + tid;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) mine[(i * TN + j) * kQuadThreads] = acc[i][j];
    } else if constexpr (HEADS) {
      // ---- element e of lane (lr, lg) of accumulator (i, 2 u + h): row i * 16 + lr, column 16 (unit % 4) + 64 h + L.lg * 4 + e of the unit's head
      const Lane L = lane_now();
      const MfmaArgs& a = args.a[cur.pi];
      const ExpandEpi& ep = args.ep[cur.pi];
      Rows late_rows;
      const Rows& R = EARLY ? early_rows : late_rows;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        if constexpr (!EARLY) {
          if (i % G == 0) request_rows(L, i, late_rows);
        }
        const int m = cur.m0 + wm * 16 * TM + i * 16 + L.lr, mc = min(m, a.B - 1), b = mc / ep.M, tok = mc - b * ep.M;
        const int slot = ep.dst_by_position ? R.pos[i % G] : tok;
        const bool keep = m < a.B && slot >= 0 && slot < ep.dst_rows;            // outside the destination: dropped
        uint16_t* row = a.y + (int64_t)b * ep.sy_b + (int64_t)slot * ep.sy_m;
        uint32_t o[U][2][2];                         // [unit][half][word]
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int unit = cur.n0 / 32 + wn * U + u, head = unit >> 2, d = (unit & 3) * 16 + L.lg * 4;
          const bool real = head * 128 < a.N;
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            float x0 = acc[i][2 * u][2 * w], x1 = acc[i][2 * u][2 * w + 1], z0 = acc[i][2 * u + 1][2 * w], z1 = acc[i][2 * u + 1][2 * w + 1];
            if (a.bias && real) {
              const uint16_t* bp = a.bias + head * 128 + d + 2 * w;
              x0 += E::val(bp[0]); x1 += E::val(bp[1]); z0 += E::val(bp[64]); z1 += E::val(bp[65]);
            }
            const uint32_t p0 = E::pack2(x0, x1), p1 = E::pack2(z0, z1);         // the projection's own rounding point
            o[u][0][w] = p0;
            o[u][1][w] = p1;
            if (ep.cos) {                            // eager 16-bit arithmetic, one rounding per op
              const uint32_t c = w ? R.cr[i % G][u].y : R.cr[i % G][u].x, sn = w ? R.sr[i % G][u].y : R.sr[i % G][u].x;
              const uint32_t q0 = E::pack2(E::lo(p0) * E::lo(c), E::hi(p0) * E::hi(c)), q1 = E::pack2(E::lo(p1) * E::lo(sn), E::hi(p1) * E::hi(sn));
              const uint32_t r0 = E::pack2(E::lo(p1) * E::lo(c), E::hi(p1) * E::hi(c)), r1 = E::pack2(E::lo(p0) * E::lo(sn), E::hi(p0) * E::hi(sn));
              o[u][0][w] = E::pack2(E::lo(q0) - E::lo(q1), E::hi(q0) - E::hi(q1));
              o[u][1][w] = E::pack2(E::lo(r0) + E::lo(r1), E::hi(r0) + E::hi(r1));
            }
          }
        }
        if constexpr (U % 2 == 0) {
#pragma unroll
          for (int u = 0; u + 1 < U; u += 2) {
            const int unit = cur.n0 / 32 + wn * U + u, head = unit >> 2;
            uint16_t* dst = row + (int64_t)head * ep.sy_h + ((unit & 3) + L.tj) * 16 + L.c8;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              quad_swap_rows(o[u][h][0], o[u + 1][h][0]);
              quad_swap_rows(o[u][h][1], o[u + 1][h][1]);
              if (keep && head * 128 < a.N) *reinterpret_cast<u32x4_any_t*>(dst + h * 64) = u32x4_t{o[u][h][0], o[u][h][1], o[u + 1][h][0], o[u + 1][h][1]};
            }
          }
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int unit = cur.n0 / 32 + wn * U + u, head = unit >> 2;
            uint16_t* dst = row + (int64_t)head * ep.sy_h + (unit & 3) * 16 + L.lg * 4;
#pragma unroll
            for (int h = 0; h < 2; ++h)
              if (keep && head * 128 < a.N) *reinterpret_cast<u32x2_any_t*>(dst + h * 64) = u32x2_t{o[u][h][0], o[u][h][1]};
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // ---- element e of lane (lr, lg) of accumulator (i, j): row i * 16 + lr, column j * 16 + L.lg * 4 + e.  Two neighbouring
      // column tiles at a time: after the swap a lane holds eight consecutive columns, tile j + tj, from c8 on.
      const Lane L = lane_now();
      const MfmaArgs& a = args.a[0];
      const int r0 = cur.m0 + wm * 16 * TM + L.lr, nb = cur.n0 + wn * 16 * TN;
      const bool res = EPI == kQuadPlain && a.res != nullptr;
      const auto word = [&](int i, int j, uint32_t (&o)[2], const float (&bz)[4]) {
        const f32x4_t v = acc[i][j];
        if constexpr (PAIR) {
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const uint32_t sg = act[PAIR ? i : 0][PAIR ? j : 0][w], uw = E::pack2(v[2 * w], v[2 * w + 1]);
            o[w] = E::pack2(E::lo(sg) * E::lo(uw), E::hi(sg) * E::hi(uw));
          }
        } else {
          o[0] = E::pack2(v[0] + bz[0], v[1] + bz[1]);
          o[1] = E::pack2(v[2] + bz[2], v[3] + bz[3]);
        }
      };
      const auto bias4 = [&](int j, float (&bz)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) bz[e] = EPI == kQuadPlain && a.bias ? E::val(a.bias[min(nb + j * 16 + L.lg * 4 + e, a.N - 1)]) : 0.f;
      };
      // COLS columns of a row, in words o[0 ..], from column n on; what is left of the row element by element
      const auto put = [&](int m, int n, auto& v, const auto& r) {
        constexpr int COLS = 2 * sizeof(v) / sizeof(uint32_t);
        typedef typename std::conditional<COLS == 8, u32x4_any_t, u32x2_any_t>::type any_t;
        const int left = a.N - n;
        if (m >= a.B || left <= 0) return;
        uint16_t* y = a.y + (int64_t)m * a.ldy + n;
        if (left >= COLS) {
          if (res) {
#pragma unroll
            for (int w = 0; w < COLS / 2; ++w) v[w] = E::pack2(E::lo(r[w]) + E::lo(v[w]), E::hi(r[w]) + E::hi(v[w]));
          }
          *reinterpret_cast<any_t*>(y) = v;
        } else {
          const uint16_t* rr = res ? a.res + (int64_t)m * a.ldres + n : nullptr;
#pragma unroll 1
          for (int e = 0; e < left; ++e) {
            uint32_t h = v[0];
#pragma unroll
            for (int w = 1; w < COLS / 2; ++w) h = (e >> 1) == w ? v[w] : h;
            h = (e & 1 ? h >> 16 : h) & 0xffffu;
            y[e] = rr ? (uint16_t)E::bits(E::val(rr[e]) + E::val(h)) : (uint16_t)h;
          }
        }
      };
#pragma unroll
      for (int jp = 0; jp < TN / 2; ++jp) {
        float bz[2][4];
        bias4(2 * jp, bz[0]);
        bias4(2 * jp + 1, bz[1]);
        Res now;                                     // all rows in flight at once
        if constexpr (EPI == kQuadPlain && !EARLY) {
          if (res) request(L, jp, now);
        }
        const Res& mine = EARLY ? rs[jp < RJ ? jp : 0] : now;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          uint32_t o[2][2];
          word(i, 2 * jp, o[0], bz[0]);
          word(i, 2 * jp + 1, o[1], bz[1]);
          quad_swap_rows(o[0][0], o[1][0]);
          quad_swap_rows(o[0][1], o[1][1]);
          u32x4_t v = {o[0][0], o[0][1], o[1][0], o[1][1]};
          put(r0 + i * 16, nb + (2 * jp + L.tj) * 16 + L.c8, v, mine[EPI == kQuadPlain ? i : 0]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (TN % 2 == 1) {
        const int n = nb + (TN - 1) * 16 + L.lg * 4;
        float bz[4];
        bias4(TN - 1, bz);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          uint32_t o[2];
          word(i, TN - 1, o, bz);
          u32x2_t v = {o[0], o[1]}, r = {0u, 0u};
          const int m = r0 + i * 16;
          if (res && m < a.B && n + 4 <= a.N) r = *reinterpret_cast<const u32x2_any_t*>(a.res + (int64_t)m * a.ldres + n);
          put(m, n, v, r);
        }
      }
    }
    if (!more) break;
    ti += wgs;
    cur = where(ti);
    request_early();
  }
  __builtin_amdgcn_s_waitcnt(0x0f70);                // loads that move nothing still count: none is under way when the LDS is given up
}

template <int DT, int EPI, int TM, int TN, int NSX, int NSW, int OCC, bool RAG = false, int H = 1, bool CUT = false>
static int launch_quad_t(QuadArgs& q, hipStream_t st, const char* who) {
  constexpr int BM = 32 * TM, BN = 32 * TN;
  constexpr size_t lds = (size_t)(NSX * BM + NSW * BN) * kQuadRow;
  static bool granted = false;
  if (!granted) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_quad_kernel<DT, EPI, TM, TN, NSX, NSW, OCC, RAG, H, CUT>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { set_last_error("%s: cannot reserve %zu bytes of LDS: %s", who, lds, hipGetErrorString(e)); return kErrLaunch; }
    granted = true;
  }
  if (EPI != kQuadHeads) q.nt = (q.a[0].N + BN - 1) / BN;
  q.mt = (q.a[0].B + BM - 1) / BM;
  const int64_t all = (int64_t)q.nt * q.mt * (EPI == kQuadShare ? q.shares : 1);
  const int64_t grid = quad_stream(TM, TN) ? std::min<int64_t>(all, (int64_t)OCC * compute_units()) : all;
  constexpr bool kAlone = OCC == 1 && TM == 4 && TN == 4 && (EPI == kQuadPlain || EPI == kQuadPair);      // beside the form of two workgroups per compute unit
  static constexpr FormText form = form_text(EPI == kQuadShare ? "shares " : (RAG ? "any quad " : "quad "), BM, BN,
                                             EPI == kQuadHeads ? " heads" : (EPI == kQuadPair ? (kAlone ? " pair alone" : " pair") :
                                             (H == 2 ? " halves" : (CUT ? " ranges" : (kAlone ? " alone" : "")))));
  set_last_form(form.s);
  const int parts = quad_asks(TM, TN) ? quad_ahead(q, all, (int64_t)q.mt * BM) : 0;
  hipLaunchKernelGGL((gemm_quad_kernel<DT, EPI, TM, TN, NSX, NSW, OCC, RAG, H, CUT>), dim3((unsigned)(grid + parts)), dim3(kQuadThreads), lds, st, q);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("%s: launch failed: %s", who, hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

}  // namespace fsvd
