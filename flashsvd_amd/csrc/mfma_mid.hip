// Projections and head expansions of prompts of 128 to about 3000 rows (head expansions from 16): workgroups of eight waves, one
// per output tile, operand rows straight into a ring of three to five LDS stages.  They serve a K below 320, the pair in the rounding that keeps the
// gate in 32 bits, ragged rows off the 4-byte grid, and the pairs and ragged rows that the rules of mfma_quad.hip leave here (figures there); everything
// else is ahead on the four-wave tiles.  Times below at a longer K are those by which the rules were set.
//
// Up to a few tiles per compute unit neither form beside this one fits: the two-stage tiles of mfma_gemm.hip rely on a second
// workgroup of the compute unit to cover a load distance of one step and wait out most of it, and the 256 x 256 tiles of
// mfma_big.hip leave compute units idle.  So the tile is chosen to give nearly every compute unit one, and loads run two to
// four steps ahead of the products behind a counted wait (a bare barrier, no fence).  The fragments of a slice are read while
// the slice before it multiplies; what is left as the bound is LDS traffic: a 128 x 192 step of 64 writes 40 KB and reads
// 112 KB of fragments for 768 cycles of products and takes about 2400 cycles, first loads and epilogue included (the pair
// 512 x 11008 x 1536 82 -> 49 us, 0.71 PFLOP/s; accumulators that a condition inside the loop may move cost another 10 us
// of register copies, hence two walks).
//
// LDS rows are 128 bytes (64 of K), their eight 16-byte pieces XOR-swizzled by row % 8.  KH = 2: waves 4-7 take the second half
// of every 128 of K and hand their sums to waves 0-3 through LDS at the end; sums run over K in the order of the forms of
// mfma_gemm.hip.  The gate / up pair runs its two products one after the other over the same tile.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace fsvd {

enum MidEpi { kMidPlain = 0, kMidPair = 1, kMidHeads = 2 };
constexpr int kMidThreads = 512, kMidRow = 128;

struct MidArgs {
  MfmaArgs a[3];                                     // heads: up to three expansions of the same token rows
  ExpandEpi ep[3];
  int first_head[4];
  int nt;                                            // column tiles
};

// RAG: any K, rows that start anywhere (plain and pair).  Loads that write LDS themselves want aligned addresses, so the pieces go
// through registers, two steps ahead of the two LDS stages; the steps past the last whole one are masked to the row, an even
// number of steps in all, so that stage and register set of a step are known to the compiler.
template <int DT, int EPI, int WM, int WN, int TM, int TN, int KH, int NS, bool RAG = false>
__global__ __launch_bounds__(kMidThreads, 2) void gemm_mid_kernel(MidArgs args) {
  typedef E16<DT> E;
  typedef typename E::frag_t frag_t;
  static_assert(WM * WN * KH == 8, "eight waves");
  static_assert(!RAG || (KH == 1 && NS == 2 && (EPI == kMidPlain || EPI == kMidPair)), "ragged rows: two stages, plain and pair");
  constexpr bool PAIR = EPI == kMidPair, HEADS = EPI == kMidHeads;
  constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN, LX = BM / 64, LW = BN / 64, LOADS = KH * (LX + LW);
  static_assert(BM % 64 == 0 && BN % 64 == 0 && (!HEADS || (BN == 128 && TN % 2 == 0)), "whole groups of rows per load");
  constexpr int kHalf = (BM + BN) * kMidRow, kStage = KH * kHalf;
  extern __shared__ __align__(16) unsigned char mid_smem[];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int kh = KH == 2 ? __builtin_amdgcn_readfirstlane(wave >> 2) : 0, wi = KH == 2 ? wave & 3 : wave;
  const int wm = __builtin_amdgcn_readfirstlane(wi / WN), wn = __builtin_amdgcn_readfirstlane(wi % WN);

  // every XCD takes one contiguous run of tiles, the row tiles of a column one after the other: W crosses from HBM once
  const int MT = gridDim.x / args.nt, t = xcd_run_index(blockIdx.x, gridDim.x);
  const int tn = t / MT, m0 = (t - tn * MT) * BM;
  const int pi = !HEADS ? 0 : (tn >= args.first_head[2] ? 2 : (tn >= args.first_head[1] ? 1 : 0));
  const MfmaArgs& a = args.a[pi];
  const ExpandEpi& ep = args.ep[pi];
  const int head = tn - args.first_head[pi], n0 = HEADS ? head * 128 : tn * BN;

  // ---- loads: eight threads per row, rows tid / 8 + 64 j of each operand; a lane's byte offset holds its row and piece, the K
  // step is the uniform offset.  Offsets fit 32 bits (the launcher checks), rows past the end are clamped to the last one.
  const int lrow = tid >> 3, lpiece = ((tid & 7) ^ (lrow & 7)) * 16;
  uint32_t xo[LX], wo[LW];
#pragma unroll
  for (int j = 0; j < LX; ++j) {
    const int r = min(m0 + lrow + 64 * j, a.B - 1);
    if (HEADS) {
      const int b = r / ep.M;
      xo[j] = (uint32_t)((b * ep.sp_b + (r - b * ep.M) * ep.sp_m) * 2) + lpiece;
    } else {
      xo[j] = (uint32_t)(r * a.ldx * 2) + lpiece;
    }
  }
#pragma unroll
  for (int j = 0; j < LW; ++j) wo[j] = (uint32_t)(min(n0 + lrow + 64 * j, a.N - 1) * a.ldw * 2) + lpiece;
  const int ksteps = RAG ? (a.K + 127) / 128 * 2 : a.K / (64 * KH), total = (PAIR ? 2 : 1) * ksteps;
  const uint32_t my_rows = (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 1024;
  const auto issue = [&](int s, int stage) {
    const bool second = PAIR && s >= ksteps;
    const uint16_t* xb = a.x + (second ? a.up_off : 0);
    const uint16_t* wb = second ? a.W2 : a.W;
    const int k = (second ? s - ksteps : s) * 128 * KH;
#pragma unroll
    for (int h = 0; h < KH; ++h) {
      unsigned char* dst = mid_smem + stage * kStage + h * kHalf + my_rows;
#pragma unroll
      for (int j = 0; j < LX; ++j) buffer_to_lds(xb, dst + j * 64 * kMidRow, xo[j], k + h * 128);
#pragma unroll
      for (int j = 0; j < LW; ++j) buffer_to_lds(wb, dst + (BM + j * 64) * kMidRow, wo[j], k + h * 128);
    }
  };
  const auto barrier = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // heads: position and rotation row of every row this thread will store, requested ahead of the operands (at the tile's end two
  // dependent loads had all workgroups of a compute unit wait at once: 333 rows of 96 heads at rank 1024 25.2 -> 24.0 us, 768 rows of
  // 48 heads at 512 16.8 -> 15.6)
  int brow[HEADS ? TM : 1], trow[HEADS ? TM : 1], prow[HEADS ? TM : 1];
  u32x2_t crow[HEADS ? TM : 1][HEADS ? TN / 2 : 1], srow[HEADS ? TM : 1][HEADS ? TN / 2 : 1];
  const bool tab8 = HEADS && ep.cos && ((reinterpret_cast<uintptr_t>(ep.cos) | reinterpret_cast<uintptr_t>(ep.sin)) & 7) == 0;
  if constexpr (HEADS) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = min(m0 + wm * 16 * TM + i * 16 + lr, a.B - 1);
      brow[i] = r / ep.M;
      trow[i] = r - brow[i] * ep.M;
      prow[i] = (ep.positions ? ep.positions[brow[i]] : ep.pos0) + trow[i];
      if (tab8) {
        const int64_t at = (int64_t)min(max(prow[i], 0), ep.rope_len - 1) * 64 + wn * 8 * TN + lg * 4;
#pragma unroll
        for (int j = 0; j < TN / 2; ++j) {
          crow[i][j] = *reinterpret_cast<const u32x2_t*>(ep.cos + at + j * 16);
          srow[i][j] = *reinterpret_cast<const u32x2_t*>(ep.sin + at + j * 16);
        }
      }
    }
  }

  const uint32_t fxo = kh * kHalf + (wm * 16 * TM + lr) * kMidRow;
  const uint32_t fwo = kh * kHalf + (BM + (HEADS ? wn * 8 * TN : wn * 16 * TN) + lr) * kMidRow;
  f32x4_t acc[TM][TN], gate[PAIR ? TM : 1][PAIR ? TN : 1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // fragments of slice kk (32 of K) of a stage
  struct Frags { frag_t x[TM], w[TN]; };
  const auto read = [&](Frags& f, int stage, int kk) {
    const unsigned char* base = mid_smem + stage * kStage + ((kk * 4 + lg) ^ (lr & 7)) * 16;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      f.w[j] = *reinterpret_cast<const frag_t*>(base + fwo + (HEADS ? (j < TN / 2 ? j * 16 : 64 + (j - TN / 2) * 16) : j * 16) * kMidRow);
#pragma unroll
    for (int i = 0; i < TM; ++i) f.x[i] = *reinterpret_cast<const frag_t*>(base + fxo + i * 16 * kMidRow);
    __builtin_amdgcn_sched_barrier(0);                 // requested here, not where they are used
  };
  const auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = E::mfma(f.w[j], f.x[i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  u32x4_t rx[RAG ? 2 : 1][LX], rw[RAG ? 2 : 1][LW];    // ragged: the pieces of steps s + 2 and s + 3
  const auto fetch = [&](int set, int s) {
    const bool second = PAIR && s >= ksteps;
    const int k = (second ? s - ksteps : s) * 64;
    const char* xb = reinterpret_cast<const char*>(a.x + (second ? a.up_off : 0) + k);
    const char* wb = reinterpret_cast<const char*>((second ? a.W2 : a.W) + k);
    if (k + 64 <= a.K) {
#pragma unroll
      for (int j = 0; j < LX; ++j) rx[set][j] = *reinterpret_cast<const u32x4_any_t*>(xb + xo[j]);
#pragma unroll
      for (int j = 0; j < LW; ++j) rw[set][j] = *reinterpret_cast<const u32x4_any_t*>(wb + wo[j]);
    } else {
      const int left = a.K - k - lpiece / 2;
#pragma unroll
      for (int j = 0; j < LX; ++j) rx[set][j] = load_masked_piece(reinterpret_cast<const uint16_t*>(xb + xo[j]), left, a.K);
#pragma unroll
      for (int j = 0; j < LW; ++j) rw[set][j] = load_masked_piece(reinterpret_cast<const uint16_t*>(wb + wo[j]), left, a.K);
    }
  };
  const auto park = [&](int set, int st) {
    unsigned char* dst = mid_smem + st * kStage + tid * 16;
#pragma unroll
    for (int j = 0; j < LX; ++j) *reinterpret_cast<u32x4_t*>(dst + j * 64 * kMidRow) = rx[set][j];
#pragma unroll
    for (int j = 0; j < LW; ++j) *reinterpret_cast<u32x4_t*>(dst + (BM + j * 64) * kMidRow) = rw[set][j];
  };
  constexpr int kW1 = (NS - 1) * LOADS, kW2 = (NS - 2) * LOADS;
  if constexpr (RAG) {
    fetch(0, 0);
    fetch(1, 1);
    park(0, 0);
    park(1, 1);
    if (total > 2) {
      fetch(0, 2);
      fetch(1, 3);
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
  } else {
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (s < total) issue(s, s);
    if (total >= NS) __builtin_amdgcn_s_waitcnt(0x0f70 | (kW1 & 15) | ((kW1 >> 4) << 14));
    else __builtin_amdgcn_s_waitcnt(0x0f70);
  }
  barrier();
  Frags f0, f1;
  read(f0, 0, 0);
  int stage = 0;
  const auto walk = [&](const int begin, const int end) {
    if constexpr (RAG) {
      for (int s0 = begin; s0 < end; s0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int s = s0 + u;
          read(f1, u, 1);
          multiply(f0);
          // the stage is read to its end and the other one written by this wave; behind the barrier by all of them
          __builtin_amdgcn_s_waitcnt(0xc07f);
          barrier();
          if (s + 1 < total) read(f0, u ^ 1, 0);
          if (s + 2 < total) park(u, u);
          if (s + 4 < total) fetch(u, s + 4);
          multiply(f1);
        }
      }
      return;
    }
    for (int s = begin; s < end; ++s) {
      read(f1, stage, 1);
      multiply(f0);
      // this wave has read the stage to its end, and its loads of the next one have landed (those of the one after may be under
      // way); behind the barrier that holds for all waves, and the stage is filled again
      if (s + NS - 1 < total) __builtin_amdgcn_s_waitcnt(0x0070 | (kW2 & 15) | ((kW2 >> 4) << 14));
      else __builtin_amdgcn_s_waitcnt(0x0070);
      barrier();
      if (s + NS < total) issue(s + NS, stage);
      stage = stage == NS - 1 ? 0 : stage + 1;
      if (s + 1 < total) read(f0, stage, 0);
      multiply(f1);
    }
  };
  walk(0, ksteps);
  if (PAIR) {                                          // the products of the second matrix go on where those of the first end
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        gate[PAIR ? i : 0][PAIR ? j : 0] = acc[i][j];
        acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    walk(ksteps, total);
  }

  if (KH == 2) {
    f32x4_t* ex = reinterpret_cast<f32x4_t*>(mid_smem);          // [TM * TN][256] 16-byte words, inside the stages
    __syncthreads();
    if (kh == 1) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) ex[(i * TN + j) * 256 + (tid & 255)] = acc[i][j];
    }
    __syncthreads();
    if (kh == 1) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += ex[(i * TN + j) * 256 + (tid & 255)];
  }

  // ---- element e of lane (lr, lg) of tile (i, j): row i * 16 + lr, column j * 16 + lg * 4 + e; four consecutive columns of a
  // row per lane (8-byte accesses where the addresses allow)
  const auto al8 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; };
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + wm * 16 * TM + i * 16 + lr;
    if (m >= a.B) continue;
    if constexpr (HEADS) {
      const int b = brow[i], tok = trow[i], pos = prow[i];
      const int slot = ep.dst_by_position ? pos : tok;
      if (slot < 0 || slot >= ep.dst_rows) continue;             // outside the destination: dropped
      uint16_t* dst = a.y + (int64_t)b * ep.sy_b + (int64_t)slot * ep.sy_m + (int64_t)head * ep.sy_h;
      const int tp = min(max(pos, 0), ep.rope_len - 1);
      const bool dst8 = al8(dst);
#pragma unroll
      for (int j = 0; j < TN / 2; ++j) {
        const int d0 = wn * 8 * TN + j * 16 + lg * 4;
        uint32_t o0[2], o1[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          const int d = d0 + 2 * w;
          float x0 = acc[i][j][2 * w], x1 = acc[i][j][2 * w + 1], z0 = acc[i][j + TN / 2][2 * w], z1 = acc[i][j + TN / 2][2 * w + 1];
          if (a.bias) {
            x0 += E::val(a.bias[head * 128 + d]); x1 += E::val(a.bias[head * 128 + d + 1]);
            z0 += E::val(a.bias[head * 128 + d + 64]); z1 += E::val(a.bias[head * 128 + d + 65]);
          }
          const uint32_t p0 = E::pack2(x0, x1), p1 = E::pack2(z0, z1);     // the projection's own rounding point
          o0[w] = p0; o1[w] = p1;
          if (ep.cos) {                                          // eager 16-bit arithmetic, one rounding per op
            uint32_t c = w ? crow[i][j].y : crow[i][j].x, sn = w ? srow[i][j].y : srow[i][j].x;
            if (!tab8) {
              const uint16_t* cp = ep.cos + (int64_t)tp * 64 + d;
              const uint16_t* sp = ep.sin + (int64_t)tp * 64 + d;
              c = cp[0] | ((uint32_t)cp[1] << 16);
              sn = sp[0] | ((uint32_t)sp[1] << 16);
            }
            const uint32_t q0 = E::pack2(E::lo(p0) * E::lo(c), E::hi(p0) * E::hi(c)), q1 = E::pack2(E::lo(p1) * E::lo(sn), E::hi(p1) * E::hi(sn));
            const uint32_t r0 = E::pack2(E::lo(p1) * E::lo(c), E::hi(p1) * E::hi(c)), r1 = E::pack2(E::lo(p0) * E::lo(sn), E::hi(p0) * E::hi(sn));
            o0[w] = E::pack2(E::lo(q0) - E::lo(q1), E::hi(q0) - E::hi(q1));
            o1[w] = E::pack2(E::lo(r0) + E::lo(r1), E::hi(r0) + E::hi(r1));
          }
        }
        if (dst8) {
          *reinterpret_cast<u32x2_t*>(dst + d0) = u32x2_t{o0[0], o0[1]};
          *reinterpret_cast<u32x2_t*>(dst + d0 + 64) = u32x2_t{o1[0], o1[1]};
        } else {
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            dst[d0 + 2 * w] = (uint16_t)o0[w]; dst[d0 + 2 * w + 1] = (uint16_t)(o0[w] >> 16);
            dst[d0 + 64 + 2 * w] = (uint16_t)o1[w]; dst[d0 + 65 + 2 * w] = (uint16_t)(o1[w] >> 16);
          }
        }
      }
    } else {
      uint16_t* yrow = a.y + (int64_t)m * a.ldy;
      const uint16_t* rrow = !PAIR && a.res ? a.res + (int64_t)m * a.ldres : nullptr;
      const bool y8 = al8(yrow), r8 = rrow && al8(rrow);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn * 16 * TN + j * 16 + lg * 4;
        if (n >= a.N) continue;
        const bool whole = n + 3 < a.N;
        uint32_t o[2];
        if (PAIR) {
          const f32x4_t g = gate[PAIR ? i : 0][PAIR ? j : 0];
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const float u0 = acc[i][j][2 * w], u1 = acc[i][j][2 * w + 1];
            if (a.mode == 0) {
              const uint32_t gw = E::pack2(g[2 * w], g[2 * w + 1]), uw = E::pack2(u0, u1);
              const uint32_t sw = E::pack2(silu_f32(E::lo(gw)), silu_f32(E::hi(gw)));
              o[w] = E::pack2(E::lo(sw) * E::lo(uw), E::hi(sw) * E::hi(uw));
            } else {
              const float g0 = g[2 * w], g1 = g[2 * w + 1];
              o[w] = E::pack2((g0 * (1.0f / (1.0f + expf(-g0)))) * u0, (g1 * (1.0f / (1.0f + expf(-g1)))) * u1);
            }
          }
        } else {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][e] + (a.bias ? E::val(a.bias[min(n + e, a.N - 1)]) : 0.f);
          o[0] = E::pack2(v[0], v[1]);
          o[1] = E::pack2(v[2], v[3]);
          if (rrow) {
            u32x2_t r;
            if (whole && r8) {
              r = *reinterpret_cast<const u32x2_t*>(rrow + n);
            } else {
              r.x = rrow[n] | ((uint32_t)rrow[min(n + 1, a.N - 1)] << 16);
              r.y = rrow[min(n + 2, a.N - 1)] | ((uint32_t)rrow[min(n + 3, a.N - 1)] << 16);
            }
            o[0] = E::pack2(E::lo(r.x) + E::lo(o[0]), E::hi(r.x) + E::hi(o[0]));
            o[1] = E::pack2(E::lo(r.y) + E::lo(o[1]), E::hi(r.y) + E::hi(o[1]));
          }
        }
        if (whole && y8) {
          *reinterpret_cast<u32x2_t*>(yrow + n) = u32x2_t{o[0], o[1]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < a.N) yrow[n + e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
  }
}

template <int DT, int EPI, int WM, int WN, int TM, int TN, int KH, int NS, bool RAG = false>
static int launch_mid_t(MidArgs& m, hipStream_t st, const char* who) {
  static bool granted = false;
  constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  constexpr size_t lds = (size_t)NS * KH * (BM + BN) * kMidRow;
  if (!granted) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid_kernel<DT, EPI, WM, WN, TM, TN, KH, NS, RAG>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { set_last_error("%s: cannot reserve %zu bytes of LDS: %s", who, lds, hipGetErrorString(e)); return kErrLaunch; }
    granted = true;
  }
  if (EPI != kMidHeads) m.nt = (m.a[0].N + BN - 1) / BN;
  const int64_t tiles = (int64_t)m.nt * ((m.a[0].B + BM - 1) / BM);
  static constexpr FormText form = form_text(RAG ? "any ring " : "ring ", BM, BN, EPI == kMidPair ? " pair" : (EPI == kMidHeads ? " heads" : ""));
  set_last_form(form.s);
  hipLaunchKernelGGL((gemm_mid_kernel<DT, EPI, WM, WN, TM, TN, KH, NS, RAG>), dim3((unsigned)tiles), dim3(kMidThreads), lds, st, m);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("%s: launch failed: %s", who, hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

static int64_t mid_tiles(const MfmaArgs& a, int bm, int bn) { return (int64_t)((a.N + bn - 1) / bn) * ((a.B + bm - 1) / bm); }
static int64_t mid_rounds(int64_t tiles) { return (tiles + compute_units() - 1) / compute_units(); }
// true when a tiling fills `share` percent of its rounds of one tile per compute unit
static bool mid_fills(int64_t tiles, int share) { return tiles * 100 >= share * compute_units() * mid_rounds(tiles); }

enum MidForm { kMidNone = 0, kMid128x192, kMid64x192, kMid128x64Halves, kMid64x64Halves, kMid128x128 };
// us per call with weights from HBM, the other forms -> this kernel:
// The pair, 128 x 192 tiles once they fill 55 percent of their rounds: 11008 x 1536 at 333 / 512 / 640 / 768 / 1024 / 1536 / 2048
// rows 64 -> 46, 82 -> 49, 97 -> 85, 100 -> 89, 102 -> 91, 176 -> 136, 195 -> 180; 5504 x 768 at 768 / 3000 rows 37 -> 28, 111 -> 83.
// A round of them takes 47 us, one of the 256 x 256 tiles 95, so those stay where they need less than half as many rounds
// (1280 rows: 101 there, 130 here).  Fewer rows: 64 x 192 tiles that fill 60 percent (11008 x 1536 at 154 / 256 rows 41 -> 35,
// 49 -> 38, 5504 x 768 at 512 26.5 -> 21.2; at 128 rows, 116 tiles, 36.6 against 37.5).
// A single matrix: 128 x 128 tiles for 144 to 256 of them (4096 x 1536 at 768 / 1024 rows 22.3 -> 18.7, 23.7 -> 20.2, 3072 x 4096 at
// 1280 49 -> 44, 2048 x 1024 at 1536 16.9 -> 13.8; two rounds of them are no better than two workgroups per compute unit:
// 4096 x 1536 at 1536 rows 33 against 37).  Below, with K halved between two groups of waves: 128 x 64 tiles for 129 to 256 of
// them (4096 x 1024 at 333 / 512 rows 12.3 -> 10.2, 12.9 -> 11.3, 3072 x 4096 at 420 29.3 -> 25.9), then 64 x 64 (4096 x 1024 at 154
// rows 8.5 -> 7.5, 1536 x 2048 at 256 15.4 -> 12.1; 64 to 128 tiles only for a short K, beyond that a K split over workgroups wins:
// 4096 x 4096 at 128 rows 18.0 against 21.9).  A K of 8192 and more is better split as well (1536 x 11008 at 512 rows 47, here 51).
// The counts are those of 256 compute units, the rules fractions of them.
static MidForm mid_form(const MfmaArgs& a, bool dual) {
  if (a.B < 128 || compute_units() <= 0 || a.K < 64 || a.K % 64 || a.ldx % 8 || a.ldw % 8 || a.up_off % 8 || !aligned16(a.x) || !aligned16(a.W) ||
      (dual && !aligned16(a.W2)) || !below_4gib(a.B, a.ldx) || !below_4gib(a.N, a.ldw))
    return kMidNone;
  if (dual) {
    const int64_t t = mid_tiles(a, 128, 192);
    if (gemm_big_apply(a, true)) return mid_rounds(t) <= 2 * mid_rounds(mid_tiles(a, 256, 256)) ? kMid128x192 : kMidNone;
    if (mid_fills(t, 55)) return kMid128x192;
    return mid_fills(mid_tiles(a, 64, 192), 60) ? kMid64x192 : kMidNone;
  }
  const int64_t big = mid_tiles(a, 128, 128), half = mid_tiles(a, 128, 64), small = mid_tiles(a, 64, 64), cu = compute_units();
  if (big * 16 >= cu * 9 && big <= cu) return kMid128x128;
  if (a.K % 128 || a.K >= 8192) return kMidNone;
  if (half * 2 > cu && half <= cu) return kMid128x64Halves;
  return small <= cu && (small * 2 > cu || (small * 4 >= cu && a.K <= 2048)) ? kMid64x64Halves : kMidNone;
}
bool gemm_mid_apply(const MfmaArgs& a, bool dual) { return mid_form(a, dual) != kMidNone; }
bool gemm_mid_pair_of_64(const MfmaArgs& a) { return mid_form(a, true) == kMid64x192; }
RingRule gemm_mid_rule(const MfmaArgs& a) {
  switch (mid_form(a, false)) {
    case kMid128x128: return RingRule{128 * 128, false};
    case kMid128x64Halves: return RingRule{128 * 64, true};
    case kMid64x64Halves: return RingRule{64 * 64, true};
    default: return RingRule{0, false};
  }
}

template <int DT>
static int launch_gemm_mid_dt(const MfmaArgs& a, bool dual, hipStream_t st, const char* who) {
  MidArgs m{};
  m.a[0] = a;
  switch (mid_form(a, dual)) {
    case kMid128x192: return launch_mid_t<DT, kMidPair, 2, 4, 4, 3, 1, 4>(m, st, who);
    case kMid64x192: return launch_mid_t<DT, kMidPair, 2, 4, 2, 3, 1, 5>(m, st, who);
    case kMid128x64Halves: return launch_mid_t<DT, kMidPlain, 2, 2, 4, 2, 2, 3>(m, st, who);
    case kMid64x64Halves: return launch_mid_t<DT, kMidPlain, 2, 2, 2, 2, 2, 4>(m, st, who);
    default: return launch_mid_t<DT, kMidPlain, 2, 4, 4, 2, 1, 4>(m, st, who);
  }
}
int launch_gemm_mid(const MfmaArgs& a, bool dual, hipStream_t st, const char* who) {
  return a.dt == 1 ? launch_gemm_mid_dt<1>(a, dual, st, who) : launch_gemm_mid_dt<0>(a, dual, st, who);
}

// Ragged rows of 128 and more.  us with weights from HBM, the two-stage tiles of mfma_gemm.hip -> this:
// The pair by the fills of the aligned one: 128 x 192 tiles, 11008 x 1492 at 333 / 512 / 768 / 1024 / 1500 rows 82 -> 65, 126 -> 67, 151 ->
// 125, 172 -> 125, 240 -> 185, 5504 x 746 at 768 / 1024 57 -> 38, 68 -> 39; 64 x 192, 11008 x 1492 at 154 / 200 56 -> 52, 56 -> 50 (128 rows, 116
// tiles, 52 against 57), 5504 x 746 at 333 / 512 32 -> 28, 42 -> 30 (aligned rows, 1536 and 768: 48, 49, 84, 92 and 28, 29).  What is left of
// the difference is pieces that straddle cache lines and their way through registers.
// A single matrix: 128 x 128 tiles for 144 to 256 of them, 4096 x 1492 at 768 / 1024 rows 30 -> 27, 33 -> 27, 3000 x 1001 at 768 25 -> 19,
// 2048 x 746 at 1500 18 -> 13 (more than a round of them, 1500 x 4096 x 1492, 42 against 50); 64 x 128 likewise, 4096 x 1492 at 512
// 22 -> 20, 3000 x 1001 at 333 / 512 17 -> 14, 19 -> 14, 2048 x 746 at 768 / 1024 12 -> 10, 13 -> 10, above a K of 2048 from seven eighths of
// a round on (4096 x 2390 at 512 rows, 256 tiles, 31 -> 30; at 333, 192 tiles, 27 against 28).
enum RagForm { kRagNone = 0, kRag128x192, kRag64x192, kRag128x128, kRag64x128 };
static RagForm mid_ragged_form(const MfmaArgs& a, bool dual) {
  const int64_t cu = compute_units();
  if (a.B < 128 || cu <= 0 || a.K < 128 || !below_4gib(a.B, a.ldx) || !below_4gib(a.N, a.ldw)) return kRagNone;     // two whole steps at least
  if (dual) return mid_fills(mid_tiles(a, 128, 192), 55) ? kRag128x192 : (mid_fills(mid_tiles(a, 64, 192), 60) ? kRag64x192 : kRagNone);
  const auto about_one = [&](int64_t t) { return t * 16 >= cu * 9 && t <= cu; };
  if (about_one(mid_tiles(a, 128, 128))) return kRag128x128;
  const int64_t t = mid_tiles(a, 64, 128);
  return about_one(t) && (a.K <= 2048 || t * 8 >= cu * 7) ? kRag64x128 : kRagNone;
}
bool gemm_mid_ragged_apply(const MfmaArgs& a, bool dual) { return mid_ragged_form(a, dual) != kRagNone; }
int gemm_mid_ragged_rows(const MfmaArgs& a) {
  const RagForm f = mid_ragged_form(a, false);
  return f == kRag64x128 ? 64 : (f == kRag128x128 ? 128 : 0);
}
template <int DT>
static int launch_mid_ragged_dt(const MfmaArgs& a, bool dual, hipStream_t st, const char* who) {
  MidArgs m{};
  m.a[0] = a;
  switch (mid_ragged_form(a, dual)) {
    case kRag128x192: return launch_mid_t<DT, kMidPair, 2, 4, 4, 3, 1, 2, true>(m, st, who);
    case kRag64x192: return launch_mid_t<DT, kMidPair, 2, 4, 2, 3, 1, 2, true>(m, st, who);
    case kRag128x128: return launch_mid_t<DT, kMidPlain, 2, 4, 4, 2, 1, 2, true>(m, st, who);
    default: return launch_mid_t<DT, kMidPlain, 2, 4, 2, 2, 1, 2, true>(m, st, who);
  }
}
int launch_mid_ragged(const MfmaArgs& a, bool dual, hipStream_t st, const char* who) {
  return a.dt == 1 ? launch_mid_ragged_dt<1>(a, dual, st, who) : launch_mid_ragged_dt<0>(a, dual, st, who);
}

// Head expansions that the 256 x 256 tiles do not take: 64 rows of a head per tile, two workgroups per compute unit (us for q, k
// and v of 32 heads at rank 1024, 64- or 128-row tiles of two stages -> this kernel: 16 rows 11.8 -> 10.6, 154 19.2 -> 15.6, 512
// 30.1 -> 25.7, 768 41.8 -> 37.1; with 8 kv heads at 333 18.6 -> 15.3; 128 or 256 rows per tile: 30.6, 28.1 at 512).  More than two tiles
// per compute unit: two stages instead of three, so that three workgroups fit one (three / two stages with weights from HBM: 333 and
// 512 rows of 96 heads at rank 1024 27.1 / 25.2, 29.9 / 28.3, at 1664 37.9 / 35.8, 42.7 / 39.4, 768 and 1024 rows of 48 heads at 512
// 18.4 / 16.8, 20.5 / 18.3; with fewer tiles the longer distance wins: 154 rows of 96 heads 18.0 / 20.0, 77 13.1 / 17.5).
bool expand_mid_apply(const ExpandArgs* d, int n) {
  for (int k = 0; k < n; ++k) {
    const ExpandArgs& a = d[k];
    if (a.R < 64 || a.R % 64 || a.sp_b % 8 || a.sp_m % 8 || a.ldu % 8 || !aligned16(a.p) || !aligned16(a.u) || a.sp_b < 0 || a.sp_m < 0 ||
        ((a.B - 1) * a.sp_b + (a.M - 1) * a.sp_m + a.R) * 2 >= (int64_t)4 << 30 || !below_4gib((int64_t)a.heads * 128, a.ldu))
      return false;
  }
  return true;
}
int launch_expand_mid(const ExpandArgs* d, int n, hipStream_t st) {
  MidArgs m{};
  const int rows = d[0].B * d[0].M;
  int heads = 0;
  for (int k = 0; k < n; ++k) {
    const ExpandArgs& a = d[k];
    m.a[k] = MfmaArgs{a.p, 0, 0, a.u, nullptr, a.ldu, a.bias, nullptr, 0, a.y, 0, rows, a.heads * 128, a.R, 0};
    m.ep[k] = ExpandEpi{a.cos, a.sin, a.rope_len, a.positions, a.M, a.sp_b, a.sp_m, a.sy_b, a.sy_m, a.sy_h, a.dst_by_position, a.dst_rows, a.pos0};
    m.first_head[k] = heads;
    heads += a.heads;
  }
  for (int k = n; k < 4; ++k) m.first_head[k] = heads;
  m.nt = heads;
  const char* who = "fsvd_lowrank_expand_heads";
  // more than two tiles per compute unit: a ring of two stages, so that three workgroups share one
  if ((int64_t)heads * ((rows + 63) / 64) > 2 * compute_units())
    return d[0].dt == 1 ? launch_mid_t<1, kMidHeads, 4, 2, 1, 4, 1, 2>(m, st, who) : launch_mid_t<0, kMidHeads, 4, 2, 1, 4, 1, 2>(m, st, who);
  return d[0].dt == 1 ? launch_mid_t<1, kMidHeads, 4, 2, 1, 4, 1, 3>(m, st, who) : launch_mid_t<0, kMidHeads, 4, 2, 1, 4, 1, 3>(m, st, who);
}

}  // namespace fsvd
