// Projections of long prompts: 256 x 256 output tiles, one workgroup of eight waves per compute unit that walks its share of
// the tiles.  They serve a K below 320; the rest runs on the tiles of mfma_quad.hip, whose four waves are ahead (q, k and v of 32 heads at 16384 x 1664
// 696 -> 594 us) or as fast (the pair 16384 x 11008 x 2432 1602 and 1605).
//
// What bounds a large product on this chip is cycles and clock alike: under a stream of these products the clock stays at 1.95 to
// 2.2 GHz (1.65 in the first milliseconds of a burst), the matrix cores are busy in 50 to 63 % of the cycles (counters), and
// every byte that has to be moved to feed the products costs both.  So the tile is the largest that one compute unit can
// hold.  A wave owns 128 x 64 of it (16 x 16 x 32 products, 128 accumulators): a K slice of 32 costs 12 fragment reads
// from LDS for 32 products, two thirds of what a 64 x 64 block costs.  K goes in steps of 64, i.e. whole
// 128-byte cache lines of every operand row (in steps of 32 every line crossed from L2 twice, because the L1 does not keep
// its other half until the next step: the loads alone then took 430 us of a 546 us product).  Loads write LDS directly, one
// step ahead into the other of two stages (two steps ahead for x, 160 KB of LDS: no faster).
//
// The two waves of a SIMD alternate: waves 0-3 (the upper half of the tile) read the fragments of a slice while waves 4-7
// multiply theirs, then the other way round, a bare barrier between the turns (published as "ping-pong" scheduling for this
// family of chips) and the multiplying wave at raised priority (12 % slower without).  A step, 2048
// cycles of products, takes 3260 to 3340 with its share of the epilogue (a single matrix, K = 4096 and 1664; 4040 for the pair);
// four waves of 128 x 128, which read a third less from LDS, were no
// faster in this turn-taking (with reads and loads laid out between their own products they are: mfma_quad.hpp).
//
// The walk over the tiles is one stream: the first stage of the next tile is requested during the last step of this one, and
// a finished tile leaves from the accumulators (pairs of 8-byte pieces become 16-byte ones by a row swap between lanes)
// while the loads are in flight and the other half of the waves still multiplies.
//
// LDS rows are 128 bytes, their eight 16-byte pieces XOR-swizzled by row % 8 (see mfma_gemm.hip).  The products run over K
// in the order of the other tiled kernels and give the same bits.  The gate / up pair runs its two products one after the
// other (SwiGLU needs nothing of the first but the gate's rounded activation, kept as packed 16-bit values); the head
// expansion takes two heads per tile, a wave the columns [32 c, 32 c + 32) and [64 + 32 c, ...) of one, so that a rotation
// pair sits in one lane.
//
// Measured with weights from HBM, 128-wide tiles -> this kernel: 16384 x 4992 x 4096 654 -> 513 us (1.31 PFLOP/s), 16384 x 4096
// x 1664 245 -> 200, the pair 16384 x 11008 x 2432 2193 -> 1533 (1.14 PFLOP/s), q, k and v of 32 heads at 16384 x 1664 842 -> 696.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace fsvd {

constexpr int kBigThreads = 512;
constexpr int kBigT = 256;                          // tile rows and columns
enum BigEpi { kBigPlain = 0, kBigPair = 1, kBigHeads = 2 };
constexpr int kBigRow = 128;                        // bytes of an operand row per K step of 64
constexpr int kBigStage = 2 * kBigT * kBigRow;      // x rows, then W rows
constexpr size_t kBigLds = (size_t)2 * kBigStage;

struct BigProblem {
  const uint16_t* x; int64_t ldx;                  // heads: rows by (batch, token), see below
  const uint16_t* W; const uint16_t* W2; int64_t ldw; int64_t up_off;
  const uint16_t* bias; const uint16_t* res; int64_t ldres;
  uint16_t* y; int64_t ldy;
  int N, K;
  // head expansion
  const uint16_t* cos; const uint16_t* sin; int rope_len;
  const int32_t* positions;
  int M; int64_t sp_b, sp_m, sy_b, sy_m, sy_h;
  int dst_by_position, dst_rows, pos0;
};
struct BigArgs { BigProblem p[3]; int first_tile[4]; int rows, nt; };   // column tiles of problem i: [first_tile[i], first_tile[i + 1])

// two tiles' words of a row of 16 lanes become consecutive words: lanes of even rows get columns 4 r .. 4 r + 7 of tile a,
// lanes of odd rows of tile b (r the row below): 8-byte pieces of two neighbouring tiles leave as 16-byte stores
__device__ __forceinline__ void swap_rows(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

template <int DT, int EPI>
__global__ __launch_bounds__(kBigThreads, 2) void gemm_big_kernel(BigArgs args) {
  typedef E16<DT> E;
  typedef typename E::frag_t frag_t;
  constexpr bool PAIR = EPI == kBigPair, HEADS = EPI == kBigHeads;
  extern __shared__ __align__(16) unsigned char big_smem[];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int wm = __builtin_amdgcn_readfirstlane(wave >> 2), wn = __builtin_amdgcn_readfirstlane(wave & 3);
  const int NT = args.nt, MT = (args.rows + kBigT - 1) / kBigT, tiles = NT * MT;
  // Every XCD takes one contiguous run of tiles in bands of eight row tiles walked column by column, its workgroups
  // neighbouring tiles of it at a time, so that they share their x and W tiles in one L2.
  const int xcd = blockIdx.x & 7, per = tiles >> 3, rem = tiles & 7;
  const int run0 = xcd * per + min(xcd, rem), run_n = per + (xcd < rem ? 1 : 0);
  const int wgs = (gridDim.x - xcd + 7) >> 3;        // workgroups of this XCD
  struct Where { int pi, m0, n0; };
  const auto where = [&](int i) {
    const int t = run0 + i, band = t / (8 * NT), tb = t - band * 8 * NT, bh = min(8, MT - band * 8);
    const int col = tb / bh;
    Where w;
    w.pi = !HEADS ? 0 : (col >= args.first_tile[2] ? 2 : (col >= args.first_tile[1] ? 1 : 0));
    w.m0 = (band * 8 + tb - col * bh) * kBigT;
    w.n0 = (col - args.first_tile[w.pi]) * kBigT;
    return w;
  };
  int ti = blockIdx.x >> 3;
  if (ti >= run_n) return;

  // ---- loads: eight threads per row, rows tid / 8 + 64 j of each operand, as buffer loads: a lane's byte offset holds its row
  // and piece, the K step is the uniform offset, so a load costs no address arithmetic and no address registers.  Offsets
  // fit 32 bits (the launcher checks), rows past the end are clamped to the last one.
  const int lrow = tid >> 3, lpiece = ((tid & 7) ^ (lrow & 7)) * 16;
  uint32_t xo[4], wo[4];
  const auto aim = [&](const Where& w) {
    const BigProblem& a = args.p[w.pi];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int xr = min(w.m0 + lrow + 64 * j, args.rows - 1);
      if (HEADS) {
        const int b = xr / a.M;
        xo[j] = (uint32_t)((b * a.sp_b + (xr - b * a.M) * a.sp_m) * 2) + lpiece;
      } else {
        xo[j] = (uint32_t)(xr * a.ldx * 2) + lpiece;
      }
      wo[j] = (uint32_t)(min(w.n0 + lrow + 64 * j, a.N - 1) * a.ldw * 2) + lpiece;
    }
  };
  const uint32_t my_rows = (uint32_t)__builtin_amdgcn_readfirstlane(wave) * 1024;      // eight rows per wave and load
  const auto issue = [&](const BigProblem& a, int s, int stage) {
    const int lsteps = a.K >> 6;
    const bool second = PAIR && s >= lsteps;
    const int k = (second ? s - lsteps : s) * 128;
    const uint16_t* xb = a.x + (second ? a.up_off : 0);
    const uint16_t* wb = second ? a.W2 : a.W;
    unsigned char* dst = big_smem + stage * kBigStage + my_rows;
#pragma unroll
    for (int j = 0; j < 4; ++j) buffer_to_lds(xb, dst + j * 64 * kBigRow, xo[j], k);
#pragma unroll
    for (int j = 0; j < 4; ++j) buffer_to_lds(wb, dst + (kBigT + j * 64) * kBigRow, wo[j], k);
  };
  const auto barrier = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ---- fragments: tiles of 16 rows 2 KB apart, piece kk * 4 + lg of a row at that piece ^ row % 8
  const uint32_t fxo = (wm * 128 + lr) * kBigRow, fwo = (kBigT + (HEADS ? (wn >> 1) * 128 + (wn & 1) * 32 : wn * 64) + lr) * kBigRow;
  Where cur = where(ti);
  aim(cur);
  issue(args.p[cur.pi], 0, 0);
  __builtin_amdgcn_s_waitcnt(0x0f70);                // the load counter only
  barrier();
  if (wm == 1) barrier();                            // half a K slice behind from here on
  int stage = 0;
  for (;;) {
    const int total = (PAIR ? 2 : 1) * (args.p[cur.pi].K >> 6), ksteps = args.p[cur.pi].K >> 6;
    const bool more = ti + wgs < run_n;
    Where nxt = cur;
    f32x4_t acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    uint32_t act[PAIR ? 8 : 1][PAIR ? 4 : 1][2];     // the pair: silu(gate), rounded, two to a word
    for (int s = 0; s < total; ++s) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        // ---- this group reads while the other multiplies
        if (kk == 0) {                               // the other stage: both groups have read it to the end
          const bool last = s + 1 == total;
          if (last && more) {
            nxt = where(ti + wgs);
            aim(nxt);
          }
          if (!last || more) issue(args.p[nxt.pi], last ? 0 : s + 1, stage ^ 1);
        }
        const uint32_t st = stage * kBigStage + (((kk * 4 + lg) ^ (lr & 7)) * 16);
        frag_t fx[8], fw[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          fw[j] = *reinterpret_cast<const frag_t*>(big_smem + st + fwo + (HEADS ? (j < 2 ? j * 16 : 64 + (j - 2) * 16) : j * 16) * kBigRow);
#pragma unroll
        for (int i = 0; i < 8; ++i) fx[i] = *reinterpret_cast<const frag_t*>(big_smem + st + fxo + i * 16 * kBigRow);
        // this slice's fragments are in registers; before the stage ends, the next one has landed
        if (kk == 1) __builtin_amdgcn_s_waitcnt(0x0070);
        else __builtin_amdgcn_s_waitcnt(0xc07f);
        barrier();
        // ---- and multiplies while the other reads
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i][j] = E::mfma(fw[j], fx[i], acc[i][j]);
        __builtin_amdgcn_s_setprio(0);
        if (PAIR && kk == 1 && s + 1 == ksteps) {
#pragma unroll
          for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
              for (int w = 0; w < 2; ++w) {
                const uint32_t g = E::pack2(acc[i][j][2 * w], acc[i][j][2 * w + 1]);
                act[i][j][w] = E::pack2(silu_f32(E::lo(g)), silu_f32(E::hi(g)));
              }
              acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        barrier();
      }
      stage ^= 1;
    }

    // ---- the finished tile: element e of lane (lr, lg) of tile (i, j) is row i * 16 + lr, column j * 16 + lg * 4 + e.  Two
    // neighbouring tiles at a time: after the swap a lane holds eight consecutive columns, tile j + (lg & 1), from
    // (lg >> 1) * 8 on.
    const BigProblem& a = args.p[cur.pi];
    const int tj = lg & 1, c8 = (lg >> 1) * 8;
    if constexpr (HEADS) {
      const int head = (cur.n0 >> 7) + (wn >> 1);
      if (head * 128 < a.N) {
        const int dc = (wn & 1) * 32;                // this wave's columns: dc .. dc + 31 and 64 past them
        float bz[2][2][4] = {};
        if (a.bias) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int e = 0; e < 4; ++e) bz[h][j][e] = E::val(a.bias[head * 128 + h * 64 + dc + j * 16 + lg * 4 + e]);
        }
        // The projection's own rounding point first: it frees half of the accumulators' registers for the rotation rows of all
        // sixteen-row tiles, which are requested at once, behind the positions of all of them (row by row, two dependent reads
        // each: the stores of a row keep the compiler from requesting the next one's before them).  q, k and v of 32 heads: 4096 rows at
        // rank 1024, an attention call on coefficients 212.6 -> 207.2 us; 16384 rows at 1664, a layer of the prompt 36 us less.  With the
        // accumulators kept in 32 bits two rows ahead were already spilled; this takes 222 registers, row by row 240.
        uint32_t o[8][2][2][2];                      // [row tile][half][tile j][word]
        int pos[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int mc = min(cur.m0 + wm * 128 + i * 16 + lr, args.rows - 1), b = mc / a.M;
          pos[i] = (a.positions ? a.positions[b] : a.pos0) + mc - b * a.M;
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const f32x4_t& v = acc[i][j + 2 * h];
              o[i][h][j][0] = E::pack2(v[0] + bz[h][j][0], v[1] + bz[h][j][1]);
              o[i][h][j][1] = E::pack2(v[2] + bz[h][j][2], v[3] + bz[h][j][3]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (a.cos) {                                 // eager 16-bit arithmetic, one rounding per op
          u32x2_t cr[8][2], sr[8][2];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int64_t at = (int64_t)min(max(pos[i], 0), a.rope_len - 1) * 64 + dc + lg * 4;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              cr[i][j] = *reinterpret_cast<const u32x2_t*>(a.cos + at + j * 16);
              sr[i][j] = *reinterpret_cast<const u32x2_t*>(a.sin + at + j * 16);
            }
          }
#pragma unroll
          for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int w = 0; w < 2; ++w) {
                const uint32_t c = w ? cr[i][j].y : cr[i][j].x, sn = w ? sr[i][j].y : sr[i][j].x, p0 = o[i][0][j][w], p1 = o[i][1][j][w];
                const uint32_t q0 = E::pack2(E::lo(p0) * E::lo(c), E::hi(p0) * E::hi(c)), q1 = E::pack2(E::lo(p1) * E::lo(sn), E::hi(p1) * E::hi(sn));
                const uint32_t r0 = E::pack2(E::lo(p1) * E::lo(c), E::hi(p1) * E::hi(c)), r1 = E::pack2(E::lo(p0) * E::lo(sn), E::hi(p0) * E::hi(sn));
                o[i][0][j][w] = E::pack2(E::lo(q0) - E::lo(q1), E::hi(q0) - E::hi(q1));
                o[i][1][j][w] = E::pack2(E::lo(r0) + E::lo(r1), E::hi(r0) + E::hi(r1));
              }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int m = cur.m0 + wm * 128 + i * 16 + lr;
          const int mc = min(m, args.rows - 1), b = mc / a.M, tok = mc - b * a.M;
          const int slot = a.dst_by_position ? pos[i] : tok;
          const bool keep = m < args.rows && slot >= 0 && slot < a.dst_rows;   // outside the destination: dropped
          uint16_t* dst = a.y + (int64_t)b * a.sy_b + (int64_t)slot * a.sy_m + (int64_t)head * a.sy_h + dc + tj * 16 + c8;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            swap_rows(o[i][h][0][0], o[i][h][1][0]);
            swap_rows(o[i][h][0][1], o[i][h][1][1]);
            if (keep) *reinterpret_cast<u32x4_t*>(dst + h * 64) = u32x4_t{o[i][h][0][0], o[i][h][0][1], o[i][h][1][0], o[i][h][1][1]};
          }
        }
      }
    } else {
      const int r0 = cur.m0 + wm * 128 + lr;
      // WHOLE: the tile lies inside the matrix
      const auto leave = [&](auto whole_t, auto res_t) {
        constexpr bool WHOLE = decltype(whole_t)::value, RES = decltype(res_t)::value;
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
          const int n = cur.n0 + wn * 64 + (j + tj) * 16 + c8, nleft = a.N - n;    // this lane's eight columns after the swap
          uint16_t* dst = a.y + (int64_t)r0 * a.ldy + n;
          const uint16_t* rr = RES ? a.res + (int64_t)r0 * a.ldres + n : nullptr;
          u32x4_t rs[RES && WHOLE ? 8 : 1];
          if (RES && WHOLE) {                        // all in flight at once
#pragma unroll
            for (int i = 0; i < 8; ++i) rs[RES && WHOLE ? i : 0] = *reinterpret_cast<const u32x4_t*>(rr + (int64_t)i * 16 * a.ldres);
          }
          float bz[2][4] = {};
          if (!PAIR && a.bias) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
              for (int e = 0; e < 4; ++e) bz[q][e] = E::val(a.bias[min(cur.n0 + wn * 64 + (j + q) * 16 + lg * 4 + e, a.N - 1)]);
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            uint32_t o[2][2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const f32x4_t v = acc[i][j + q];
              if (PAIR) {
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                  const uint32_t g = act[PAIR ? i : 0][PAIR ? j + q : 0][w], u = E::pack2(v[2 * w], v[2 * w + 1]);
                  o[q][w] = E::pack2(E::lo(g) * E::lo(u), E::hi(g) * E::hi(u));
                }
              } else {
                o[q][0] = E::pack2(v[0] + bz[q][0], v[1] + bz[q][1]);
                o[q][1] = E::pack2(v[2] + bz[q][2], v[3] + bz[q][3]);
              }
            }
            swap_rows(o[0][0], o[1][0]);
            swap_rows(o[0][1], o[1][1]);
            u32x4_t v = {o[0][0], o[0][1], o[1][0], o[1][1]};
            const auto add = [&](const u32x4_t& r) {
              v.x = E::pack2(E::lo(r.x) + E::lo(v.x), E::hi(r.x) + E::hi(v.x));
              v.y = E::pack2(E::lo(r.y) + E::lo(v.y), E::hi(r.y) + E::hi(v.y));
              v.z = E::pack2(E::lo(r.z) + E::lo(v.z), E::hi(r.z) + E::hi(v.z));
              v.w = E::pack2(E::lo(r.w) + E::lo(v.w), E::hi(r.w) + E::hi(v.w));
            };
            if (WHOLE) {
              if (RES) add(rs[RES && WHOLE ? i : 0]);
              *reinterpret_cast<u32x4_t*>(dst + (int64_t)i * 16 * a.ldy) = v;
              continue;
            }
            if (r0 + i * 16 >= args.rows || nleft <= 0) continue;
            uint16_t* d = dst + (int64_t)i * 16 * a.ldy;
            const uint16_t* rp = RES ? rr + (int64_t)i * 16 * a.ldres : nullptr;
            if (nleft >= 8) {
              if (RES) add(*reinterpret_cast<const u32x4_t*>(rp));
              *reinterpret_cast<u32x4_t*>(d) = v;
            } else {
              const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
              for (int e = 0; e < 7; ++e)
                if (e < nleft) {
                  const uint32_t h = (w[e >> 1] >> (16 * (e & 1))) & 0xffffu;
                  d[e] = RES ? (uint16_t)E::bits(E::val(rp[e]) + E::val(h)) : (uint16_t)h;
                }
            }
          }
        }
      };
      const bool whole = cur.m0 + kBigT <= args.rows && cur.n0 + kBigT <= a.N;
      typedef std::integral_constant<bool, true> yes_t;
      typedef std::integral_constant<bool, false> no_t;
      if (!PAIR && a.res) {
        if (whole) leave(yes_t{}, std::integral_constant<bool, !PAIR>{});
        else leave(no_t{}, std::integral_constant<bool, !PAIR>{});
      } else if (whole) {
        leave(yes_t{}, no_t{});
      } else {
        leave(no_t{}, no_t{});
      }
    }
    if (!more) break;
    cur = nxt;
    ti += wgs;
  }
  if (wm == 0) barrier();                            // the other group's last turn
}

template <int DT, int EPI>
static int launch_big_t(const BigArgs& a, hipStream_t st, const char* who) {
  static bool granted = false;
  constexpr size_t lds = kBigLds;
  if (!granted) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_big_kernel<DT, EPI>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { set_last_error("%s: cannot reserve %zu bytes of LDS: %s", who, lds, hipGetErrorString(e)); return kErrLaunch; }
    granted = true;
  }
  const int tiles = a.nt * ((a.rows + kBigT - 1) / kBigT);
  set_last_form(EPI == kBigPair ? "256 x 256 pair" : (EPI == kBigHeads ? "256 x 256 heads" : "256 x 256"));
  hipLaunchKernelGGL((gemm_big_kernel<DT, EPI>), dim3(std::min(tiles, compute_units())), dim3(kBigThreads), lds, st, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("%s: launch failed: %s", who, hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}

// Worth it when the rounds of one tile per compute unit are more than about half full (`share` percent): below that the
// smaller tiles of mfma_gemm.hip, which leave fewer compute units idle, are ahead.  us per call, those tiles -> this kernel:
// 320 tiles (8192 x 2432 x 11008, 62 % full) 557 -> 486, 448 (16384 x 1664 x 4096, 87 %) 269 -> 193, 160 (5000 x 2048 x 2048,
// 62 %) 68 -> 46, 256 (4096 x 4096 x 4096) 158 -> 105; 128 tiles (2048 x 4096 x 4096, 50 %) 80 -> 97, 96 tiles (4096 x 1536 x
// 11008, 37 %) 181 -> 243.  The gate / up pair comes here where mfma_mid.hip needs more than twice the rounds (its 128 x 192 tiles
// take half as long): 1280 rows of 11008 x 1536 (84 % of one round) 101 here and 130 there.
static bool big_worth(int64_t rows, int64_t col_tiles, int share) {
  const int64_t tiles = ((rows + kBigT - 1) / kBigT) * col_tiles, cu = compute_units();
  return rows >= kBigT && cu > 0 && tiles * 100 >= share * cu * ((tiles + cu - 1) / cu);
}

bool gemm_big_apply(const MfmaArgs& a, bool dual) {
  if (dual && a.mode != 0) return false;             // the fused rounding keeps the gate in fp32
  return big_worth(a.B, (a.N + kBigT - 1) / kBigT, dual ? 50 : 55) && a.K > 0 && a.K % 64 == 0 && a.ldx % 8 == 0 && a.ldw % 8 == 0 && a.ldy % 8 == 0 && a.up_off % 8 == 0 &&
         aligned16(a.x) && aligned16(a.W) && (!dual || aligned16(a.W2)) && aligned16(a.y) && (a.res == nullptr || (aligned16(a.res) && a.ldres % 8 == 0)) &&
         below_4gib(a.B, a.ldx) && below_4gib(a.N, a.ldw);
}
int launch_gemm_big(const MfmaArgs& m, bool dual, hipStream_t st, const char* who) {
  BigArgs a{};
  BigProblem& p = a.p[0];
  p.x = m.x; p.ldx = m.ldx; p.W = m.W; p.W2 = m.W2; p.ldw = m.ldw; p.up_off = m.up_off; p.bias = m.bias; p.res = m.res; p.ldres = m.ldres;
  p.y = m.y; p.ldy = m.ldy; p.N = m.N; p.K = m.K;
  a.rows = m.B;
  a.nt = (m.N + kBigT - 1) / kBigT;
  if (dual) return m.dt == 1 ? launch_big_t<1, kBigPair>(a, st, who) : launch_big_t<0, kBigPair>(a, st, who);
  return m.dt == 1 ? launch_big_t<1, kBigPlain>(a, st, who) : launch_big_t<0, kBigPlain>(a, st, who);
}

bool expand_big_apply(const ExpandArgs* d, int n) {
  int64_t tiles = 0;
  for (int i = 0; i < n; ++i) {
    const ExpandArgs& a = d[i];
    const auto al8 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; };
    if (a.R % 64 || a.sp_b % 8 || a.sp_m % 8 || a.ldu % 8 || a.sy_b % 8 || a.sy_m % 8 || a.sy_h % 8 || !aligned16(a.p) || !aligned16(a.u) || !aligned16(a.y) ||
        (a.cos && !(al8(a.cos) && al8(a.sin))))
      return false;
    if (a.sp_b < 0 || a.sp_m < 0 || ((a.B - 1) * a.sp_b + (a.M - 1) * a.sp_m + a.R) * 2 >= (int64_t)4 << 30 || !below_4gib((int64_t)a.heads * 128, a.ldu)) return false;
    tiles += (a.heads + 1) / 2;
  }
  return big_worth((int64_t)d[0].B * d[0].M, tiles, 65);   // q, k and v of 32 heads at 1024 rows (75 %) 42 against 44 us of 64-row tiles, at 1536 (56 %) 77 against 69
}
int launch_expand_big(const ExpandArgs* d, int n, hipStream_t st) {
  BigArgs a{};
  int tiles = 0;
  for (int i = 0; i < n; ++i) {
    const ExpandArgs& e = d[i];
    BigProblem& p = a.p[i];
    p.x = e.p; p.W = e.u; p.ldw = e.ldu; p.bias = e.bias; p.y = e.y; p.N = e.heads * 128; p.K = e.R;
    p.cos = e.cos; p.sin = e.sin; p.rope_len = e.rope_len; p.positions = e.positions; p.M = e.M; p.sp_b = e.sp_b; p.sp_m = e.sp_m;
    p.sy_b = e.sy_b; p.sy_m = e.sy_m; p.sy_h = e.sy_h; p.dst_by_position = e.dst_by_position; p.dst_rows = e.dst_rows; p.pos0 = e.pos0;
    a.first_tile[i] = tiles;
    tiles += (e.heads + 1) / 2;
  }
  for (int i = n; i < 4; ++i) a.first_tile[i] = tiles;
  a.rows = d[0].B * d[0].M;
  a.nt = tiles;
  const char* who = "fsvd_lowrank_expand_heads";
  return d[0].dt == 1 ? launch_big_t<1, kBigHeads>(a, st, who) : launch_big_t<0, kBigHeads>(a, st, who);
}

}  // namespace fsvd
