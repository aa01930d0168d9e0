// Projections of prompts on the four-wave tiles of mfma_quad.hpp: which tile a shape gets, the single matrices, the gate / up pair,
// and long K in shares over workgroups.
#include "mfma_quad.hpp"

namespace fsvd {

static int64_t quad_tiles(const MfmaArgs& a, int tm, int tn) { return (int64_t)((a.N + 32 * tn - 1) / (32 * tn)) * ((a.B + 32 * tm - 1) / (32 * tm)); }

constexpr float kLaunchUs = 3.f, kShareSumUs = 3.5f, kShareBytesPerUs = 4.5e6f;      // of a launch; of the one that adds the shares, beside their way out and in
static float share_sum_us(int64_t floats) { return kShareSumUs + (float)floats * 8.f / kShareBytesPerUs; }
#define FSVD_QUAD_PAIR(X) \
  X(0, 4, 6, 3, 4, 1, 0.f, 0.f, 8.19f, 0.657f) X(1, 5, 6, 2, 3, 1, 0.f, 0.f, 9.82f, 0.693f) X(2, 5, 4, 2, 2, 2, 4.26f, 0.861f, 8.46f, 0.970f) \
  X(3, 8, 4, 2, 3, 1, 0.f, 0.f, 10.88f, 0.710f) X(4, 4, 4, 2, 3, 2, 3.94f, 0.589f, 7.43f, 0.802f) X(5, 4, 4, 4, 5, 1, 0.f, 0.f, 6.31f, 0.487f) \
  X(6, 3, 6, 3, 4, 1, 0.f, 0.f, 6.98f, 0.562f) X(7, 3, 3, 3, 3, 2, 1.93f, 0.444f, 4.61f, 0.652f) X(8, 2, 3, 3, 4, 2, 2.96f, 0.273f, 2.34f, 0.547f) \
  X(9, 2, 2, 5, 5, 2, 1.50f, 0.330f, 1.50f, 0.490f)
// ragged rows: some of them
#define FSVD_QUAD_PLAIN_ANY(X) X(4, 6, 4, 3, 4, 1) X(5, 4, 4, 2, 3, 2) X(10, 3, 2, 3, 4, 2) X(12, 2, 2, 5, 5, 2)
#define FSVD_QUAD_PAIR_ANY(X) X(0, 4, 6, 3, 4, 1) X(4, 4, 4, 2, 3, 2) X(6, 3, 6, 3, 4, 1) X(7, 3, 3, 3, 3, 2) X(8, 2, 3, 3, 4, 2)

constexpr int kQuadNone = -1;
struct QuadPick { int form; float us; };
// The order of the sums of 128 aligned rows and more is the one that the shape had on the tiles before these (rings with K halved between waves, 64 x
// 64 tiles with K cut over workgroups), so that the bits stay: a model of 32 layers hands a flipped rounding on until another order of the same
// sums ends 0.046 (relative) away.  Both cost nothing here: a second set of accumulators, a sum kept in registers.  Other orders than before have 33
// to 127 rows (one sum, no split), ragged single matrices (one sum; the tiles before halved K between waves), a K of 4096 to 5119 that filling_shares
// declines by its costs, and a K of 8192 and more without scratch that split_is_ahead leaves here (133 such shapes: the error against
// 64 bits, 0.0017 from the output's rounding, grows by at most 1.2e-7 of itself).
enum QuadOrder { kOrderPlain = 0, kOrderHalves = 1, kOrderCut = 2 };
struct QuadSums { QuadOrder order; int per; };
static QuadSums quad_sums(const MfmaArgs& a) {
  if (a.B < 128 || gemm_big_apply(a, false)) return QuadSums{kOrderPlain, 0};
  const RingRule r = gemm_mid_rule(a);
  if (r.area > 0) return QuadSums{r.halves ? kOrderHalves : kOrderPlain, 0};
  const int per = a.K < 8192 ? gemm_tiles_cut(a).per : 0;                             // longer ones: in shares, or one sum
  return per > 0 ? QuadSums{kOrderCut, per} : QuadSums{kOrderPlain, 0};
}
static QuadPick quad_pick(const MfmaArgs& a, bool dual, bool any, QuadOrder order = kOrderPlain) {
  if (order == kOrderCut) return QuadPick{12, ranges_us(quad_tiles(a, 2, 2), a.K, compute_units())};       // few 64 x 64 tiles by that rule
  QuadPick best{kQuadNone, 0.f};
  const float steps = (float)((a.K + 63) / 64 * (dual ? 2 : 1));
  const int64_t cu = compute_units();                // asked once: a small model's call is bound by what the host does per launch
  const auto take = [&](int form, int tm, int tn, int occ, const QuadCost& c) {
    const float us = quad_us(c, quad_tiles(a, tm, tn), occ, steps, cu);
    if (best.form == kQuadNone || us < best.us) best = QuadPick{form, us};
  };
  if (dual) {
#define X(n, TM, TN, SX, SW, OCC, F1, S1, F2, S2) if (!any || n == 0 || n == 4 || (n >= 6 && n <= 8)) take(n, TM, TN, OCC, QuadCost{F1, S1, F2, S2});
    FSVD_QUAD_PAIR(X)
#undef X
  } else {
    // 96 x 64 is left out for a K of 4096 and more: 64 x 64 and 128 x 64 are within 6 % of it or ahead there (3072 columns at 154, 333,
    // 420, 512 rows 22.5, 22.2, 22.2, 27.6 against 17.9, 21.5, 23.7, 27.2), below it is the best tile of 333 rows (4096 x 1536 11.4 against
    // 12.8).  64 x 96 is a tile for one per compute unit: 512 x 2238 x 4096 28.2 -> 24.6, 511 x 3072 x 4096 28.0 -> 25.4, 192 x 7717 x 8000 48.4 -> 50.3 (0.86 to
    // 1.06 of 128 x 64 over 47 shapes); over more the others are up to 15 % ahead.
    const auto fits = [&](int n) {
      if (any) return n == 4 || n == 5 || n == 10 || n == 12;
      if (order != kOrderPlain && !quad_halves(n)) return false;
      // two row tiles of 96 and more than a column of them per compute unit: 128 x 128 is ahead of its costs there (192 x 13260 x 1536 23.0 -> 19.7, 174 x 16384
      // x 2048 30.2 -> 23.2, K 1024 as fast); 64 x 128 is a tile for one round (300 x 24000 x 320 20.5 -> 15.6, 700 x 11008 x 320 19.4 -> 14.3)
      if (n == 10 && a.B >= 128 && a.B <= 192 && a.K >= 1280 && quad_tiles(a, 3, 2) > cu) return false;
      if (n == 9 && quad_tiles(a, 2, 4) > cu) return false;
      return n == 10 ? a.K < 4096 : (n == 11 ? quad_tiles(a, 2, 3) <= cu : true);
    };
#define X(n, TM, TN, SX, SW, OCC, F1, S1, F2, S2) if (fits(n)) take(n, TM, TN, OCC, QuadCost{F1, S1, F2, S2});
    FSVD_QUAD_PLAIN(X)
#undef X
  }
  return best;
}

// rows of whole pieces that start on the 16-byte grid, K of whole steps
static bool quad_grid(const MfmaArgs& a, bool dual) {
  return a.K % 64 == 0 && a.ldx % 8 == 0 && a.ldw % 8 == 0 && a.up_off % 8 == 0 && aligned16(a.x) && aligned16(a.W) && (!dual || aligned16(a.W2));
}
// rows on the 4-byte grid, which is what a 16-byte load asks of its address
static bool quad_words(const MfmaArgs& a, bool dual) {
  const auto al4 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3) == 0; };
  return a.ldx % 2 == 0 && a.ldw % 2 == 0 && a.up_off % 2 == 0 && al4(a.x) && al4(a.W) && (!dual || al4(a.W2));
}
// From 128 rows and five K steps on (fewer steps than the stages hold are left to the tiles that were measured for them), but for what the rules in
// front of gemm_quad_apply leave to other kernels; N holds a whole residual piece.  The pair in the rounding that keeps the gate in 32 bits goes to
// mfma_mid.hip.  From 33 rows on where there are 64 tiles of 64 x 64 with a K below 4096, or 128 of them (us at 40 / 64 / 100 rows, 32-row tiles with K split over workgroups -> these: the pair 11008 x 1536 30.6 ->
// 19.3, 31.9 -> 21.4, 34.5 -> 23.3, 32000 x 4096 65 -> 53, 72 -> 56, 99 -> 62, 4096 x 1024 8.7 -> 7.4, 8.9 -> 8.2, 10.9 -> 7.5); fewer tiles
// need the split (3072 x 4096 16.1 against 18.5, 16.9 against 21.3; 1024 x 4096 9.4 against 17.8).
static bool quad_range(const MfmaArgs& a, bool dual) {
  if (a.B < 33 || a.K < 320 || a.N < 8 || compute_units() <= 0 || (dual && a.mode != 0) || !below_4gib(a.B, a.ldx) || !below_4gib(a.N, a.ldw)) return false;
  const int64_t tiles = quad_tiles(a, 2, 2), cu = compute_units();
  return a.B >= 128 || tiles * 2 >= cu || (tiles * 4 >= cu && a.K < 4096);
}

// A long K in shares over workgroups, about one workgroup of the launch per compute unit, their sums in scratch of the call's own
// (so that calls on different streams stay independent): tiles of 64 x 128 up to 192 rows, 256 x 128
// from 385 on where they pad no more rows than 128 x 128 do (768 rows of 1536 x 11008 40 us against 45), else 128 x 128 (256 rows 24
// against 27).  us with weights from HBM, what runs otherwise -> this:
// K of 8192 and more, always: 1536 x 11008 (64-row tiles of two stages whose last workgroup adds the shares) at 128 / 154 / 256 / 333 /
// 512 / 768 / 1024 rows 24 -> 20, 30 -> 24, 32 -> 24, 41 -> 28, 45 -> 36, 63 -> 45, 67 -> 47; 1536 x 8192 at 1536 / 2048 (ring of 128 x
// 128) 71 -> 53, 74 -> 69; 2390 x 11008 at 2048 (128 x 64 tiles; one share) 194 -> 161.  Where no ring takes the shape and 64- or 128-row
// tiles fill 70 percent of the compute units with it, K is cut as the 64 x 64 tiles cut it, whose bits those rows had before; as many shares
// as the chip has room for took 19, 20, 23, 26, 32, 39 at the first six of these row counts.
// K of 4096 to 8191: adding up the shares has to come out of the compute units that work here and not under the ring, i.e. out of
// gain = shares * area(ring tile) / area(tile), where area counts a workgroup's outputs.
//   gain 1.5: 128 x 4992 x 4096 22.1 -> 19.6, 333 x 3072 x 4096 25.2 -> 23.7, 768 x 3072 x 4096 38.7 -> 34.8, 1536 x 1500 x 5504 51 -> 41, 640 x 2048 x
//     5504 36 -> 28.  Taken: from 1.4 on.
//   gain 1.25, outputs for 90 percent of the compute units and more: 768 x 2048 x 5504 36 -> 32, 1024 x 1500 x 5504 37 -> 32; at a K of 4096, where
//     the sum weighs more, only 4 percent (512 x 3072 x 4096 28.9 -> 27.7).  Taken: from 1.2 on with a K of 5120 and more.
//   gain 1.25, a quarter of it padding: 420 x 3072 x 4096 24 -> 28, 200 x 3072 x 4096 17.0 -> 19.5; gain 1: 512 x 4096 x 4096 30.9 -> 31.8.  Not taken.
//   no ring to compare with: from three shares over 3/16 of the compute units on: 128 x 3072 x 4096 21 -> 16, 154 x 2048 x 5504 22 -> 17.
struct ShareForm { int bm, bn, shares, per; };
// as many shares as there are compute units for
static ShareForm filling_shares(const MfmaArgs& a, const RingRule& ring) {
  const ShareForm none{0, 0, 0, 0};
  const int64_t cu = compute_units();
  const auto pad = [&](int64_t r) { return (a.B + r - 1) / r * r; };
  const int steps = a.K / 64;
  const int bm = a.B <= 192 ? 64 : (a.B > 384 && pad(256) <= pad(128) ? 256 : 128);
  const int64_t tiles = quad_tiles(a, bm / 32, 4), area = (int64_t)bm * 128;
  int64_t shares = std::min<int64_t>(cu / tiles, steps / 8);                         // eight steps each at least
  shares = std::min<int64_t>(shares, (int64_t)(a.scratch_floats / (size_t)(tiles * area)));
  if (a.K < 8192) {
    const bool full = a.K >= 5120 && (int64_t)a.B * a.N * shares * 10 >= 9 * cu * area;
    if (ring.area == 0 ? shares < 3 || tiles * 16 < 3 * cu : shares * ring.area * 100 < (full ? 120 : 140) * area) return none;
  }
  if (shares < 1) return none;
  const int per = (steps + (int)shares - 1) / (int)shares;
  shares = (steps + per - 1) / per;
  // the sums once out and once in, and the launch that adds them; 333 x 1664 x 4096 19.7 us in shares, 16.1 unsplit (here too a K below 5120 only:
  // the longer ones were ahead in shares at every row count)
  if (a.K < 5120) {
    const float us = share_us(bm, 128, shares * tiles, per, cu) + share_sum_us(shares * tiles * area);
    if (kLaunchUs + quad_pick(a, false, false).us < 0.9f * (kLaunchUs + us)) return none;
  }
  return ShareForm{bm, 128, (int)shares, per};
}
static ShareForm share_form(const MfmaArgs& a) {
  const ShareForm none{0, 0, 0, 0};
  if (a.scratch_floats == 0 || a.B < 128 || a.K < 4096 || !quad_range(a, false) || !quad_grid(a, false) || gemm_big_apply(a, false)) return none;
  const int64_t cu = compute_units();
  const int steps = a.K / 64;
  const RingRule ring = gemm_mid_rule(a);
  // the cut of the 64 x 64 tiles, where a tile of this kernel fills 70 percent of the compute units with it: the same bits
  if (a.K >= 8192 && ring.area == 0) {
    const int per = gemm_tiles_cut(a).per;
    for (const int bm : {64, 128}) {
      const int64_t t = quad_tiles(a, bm / 32, 4) * (per ? (steps + per - 1) / per : 0);
      if (t * 10 >= 7 * cu && t <= cu && (size_t)t * bm * 128 <= a.scratch_floats) return ShareForm{bm, 128, (steps + per - 1) / per, per};
    }
  }
  const ShareForm filling = filling_shares(a, ring);
  if (filling.shares > 0) return filling;
  // K cut in ranges (see quad_sums): one workgroup per range and 64 x 64 tile where that beats one after the other (512 x 1024 x 4096 in two
  // ranges 19.6 -> 16.4 us, 154 x 1024 x 4096 in six 18.6 -> 12.1).  Shapes that fill the chip with shares of 64 x 128 do not come here (128 x 3072 x 5120
  // 16.9 us there, 24.8 in ranges, 154 x 2048 x 8064 19.3 and 26.5).  A long walk takes up to 1.2 times its costs (384 x 1300 x 5120 26.3 us), hence the 1.1.
  const QuadSums sums = quad_sums(a);
  if (sums.order != kOrderCut) return none;
  const int64_t tiles = quad_tiles(a, 2, 2), shares = (steps + sums.per - 1) / sums.per;
  const float apart = share_us(64, 64, tiles * shares, sums.per, cu) + share_sum_us(shares * tiles * 4096);
  return apart < 1.1f * ranges_us(tiles, a.K, cu) && (size_t)(tiles * shares * 4096) <= a.scratch_floats ? ShareForm{64, 64, (int)shares, sums.per} : none;
}
// floats of scratch that the call can use, out of at most `cap`
size_t gemm_share_floats(MfmaArgs a, size_t cap) {
  a.scratch_floats = cap;
  const ShareForm f = share_form(a);
  return f.shares > 0 ? (size_t)f.shares * quad_tiles(a, f.bm / 32, f.bn / 32) * f.bm * f.bn : 0;
}

// The shares of every tile, added in their order, and the epilogue of a single matrix: one thread per four columns of a row, as the
// accumulators hold them.  A launch of its own: the shares need no counters, and all compute units add.
template <int DT, int TM, int TN>
__global__ __launch_bounds__(256) void share_sum_kernel(QuadArgs args, int tiles) {
  typedef E16<DT> E;
  constexpr int kWords = TM * TN * kQuadThreads, BM = 32 * TM, BN = 32 * TN;
  const MfmaArgs& a = args.a[0];
  const int g = blockIdx.x * 256 + threadIdx.x, t = g / kWords, r = g - t * kWords;
  const f32x4_t* part = reinterpret_cast<const f32x4_t*>(args.part) + (size_t)t * args.shares * kWords + r;
  f32x4_t v = part[0];
  int z = 1;
  for (; z + 4 <= args.shares; z += 4) {               // four shares on their way at a time
    f32x4_t w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = part[(size_t)(z + u) * kWords];
#pragma unroll
    for (int u = 0; u < 4; ++u) v += w[u];
  }
  for (; z < args.shares; ++z) v += part[(size_t)z * kWords];
  const int ij = r / kQuadThreads, tid = r - ij * kQuadThreads, i = ij / TN, j = ij - i * TN, wave = tid >> 6, lane = tid & 63;
  const int NT = args.nt, band = t / (8 * NT), tb = t - band * 8 * NT, bh = min(8, args.mt - band * 8), col = tb / bh;
  const int m = (band * 8 + tb - col * bh) * BM + (wave >> 1) * 16 * TM + i * 16 + (lane & 15);
  const int n = col * BN + (wave & 1) * 16 * TN + j * 16 + (lane >> 4) * 4;
  if (m >= a.B || n >= a.N) return;
  const uint16_t* res = a.res ? a.res + (int64_t)m * a.ldres + n : nullptr;
  uint16_t* y = a.y + (int64_t)m * a.ldy + n;
  uint32_t o[2];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (a.bias && n + e < a.N) v[e] += E::val(a.bias[n + e]);
  }
  o[0] = E::pack2(v[0], v[1]);
  o[1] = E::pack2(v[2], v[3]);
  const bool whole = n + 3 < a.N;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (res && n + e < a.N) v[e] = E::val(res[e]) + E::val((o[e >> 1] >> (16 * (e & 1))) & 0xffffu);
  }
  if (res) {
    o[0] = E::pack2(v[0], v[1]);
    o[1] = E::pack2(v[2], v[3]);
  }
  if (whole && (reinterpret_cast<uintptr_t>(y) & 7) == 0) {
    *reinterpret_cast<u32x2_t*>(y) = u32x2_t{o[0], o[1]};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < a.N) y[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
  }
}
template <int DT, int TM, int TN, int NSX, int NSW, int OCC>
static int launch_share_t(QuadArgs& q, hipStream_t st, const char* who) {
  const int rc = launch_quad_t<DT, kQuadShare, TM, TN, NSX, NSW, OCC>(q, st, who);
  if (rc != kOk) return rc;
  const int tiles = q.nt * q.mt;
  hipLaunchKernelGGL((share_sum_kernel<DT, TM, TN>), dim3(tiles * TM * TN * kQuadThreads / 256), dim3(256), 0, st, q, tiles);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) { set_last_error("%s: launch failed: %s", who, hipGetErrorString(e)); return kErrLaunch; }
  return kOk;
}
template <int DT>
static int launch_share_dt(QuadArgs& q, const ShareForm& f, hipStream_t st, const char* who) {
  if (f.bn == 64) return launch_share_t<DT, 2, 2, 5, 5, 2>(q, st, who);
  if (f.bm == 64) return launch_share_t<DT, 2, 4, 3, 4, 1>(q, st, who);
  return f.bm == 128 ? launch_share_t<DT, 4, 4, 4, 5, 1>(q, st, who) : launch_share_t<DT, 8, 4, 3, 3, 1>(q, st, who);
}

// ---- what stays with the kernels before these because they are ahead there.  How full the row tiles are counts throughout: as many tiles take longer with
// full ones (64 of 256 and of 200 rows, 1024 x 3584, one per compute unit: 18.0 and 14.7 us; why is not shown yet), and more so here than there.
static bool rows_fill(const MfmaArgs& a) { return (int64_t)a.B * 16 >= (int64_t)((a.B + 63) / 64) * 64 * 15; }

// A call of 128 rows and more that runs in no shares of its own: the 64 x 64 tiles of mfma_gemm.hip, K split over workgroups that add up in the registered
// buffer, where that has room and the split is ahead of one workgroup per tile.  us in one workgroup / split, tiles x ranges in brackets,
// weights from HBM:
//   K of 1536 to 8191: up to one workgroup of the split per compute unit, 128 x 1024 x 1536 (32 x 3) 10.3 / 9.4, x 4096 (32 x 8) 19.8 / 12.4, 256 x 1024 x
//     3584 (64 x 4) 17.4 / 12.0, 512 x 1024 x 5504 (128 x 2) 26.4 / 20.5; below 2048 with full row tiles and 512 columns only (185 x 812 x 1600 10.3 /
//     11.1, 128 x 1024 x 1024 7.9 / 9.1).  More workgroups lose, as neighbours on a compute unit cover each other, 333 x 704 x 3072 (66 x 4) 13.4 / 14.6, 592 x
//     267 x 1856 (50 x 6) 9.3 / 13.9, until K is long: 128 x 1536 x 5504 (48 x 6) 26.8 / 18.7, 128 x 2560 x 3840 (80 x 4) 21.4 / 19.0, 154 x 1536 x 5504 (72 x
//     4) 22.2 / 20.2 (x 4096 17.4 / 17.9).
//   K of 8192 and more: up to 128 tiles, 128 x 1536 x 11008 51.9 / 24.6, 512 x 1024 x 8192 34.1 / 29.2, up to 192 with full row tiles from 10240 on, 512 x 1536 x
//     11008 50.9 / 46.4.  Not 200 x 2560 x 11008 (160 tiles) 39.7 / 46.6.
static bool split_is_ahead(const MfmaArgs& a) {
  if (a.B < 128 || a.K < 1536 || gemm_mid_rule(a).area > 0 || gemm_big_apply(a, false)) return false;
  const int64_t tiles = quad_tiles(a, 2, 2), cu = compute_units();
  const TilesCut c = gemm_tiles_cut(a);
  if (!c.room) return false;
  const int64_t wgs = tiles * c.ranges;
  const bool full = rows_fill(a);
  bool ahead;
  if (a.K >= 8192) ahead = tiles * 2 <= cu || (full && a.K >= 10240 && tiles * 4 <= cu * 3);
  else if (wgs <= cu) ahead = a.K >= 2048 || (full && a.N >= 512);
  else if (tiles * 5 <= cu) ahead = a.K >= (full ? 3072 : 4096);
  else ahead = a.N >= 320 && wgs * 3 <= cu * 4 && a.K >= (full ? 3584 : 5120);
  return ahead && share_form(a).shares == 0;
}

// 33 to 127 aligned rows with at most one 32 x 64 tile per compute unit: those of mfma_gemm.hip, K split over workgroups in the registered buffer, where K
// is long.  The split gives every compute unit two workgroups, or a few more and with them a second round; from which K on it is ahead goes by that
// and by how many ranges there are.  us here / split, weights from HBM: a single matrix of up to half as many tiles, 64 x 4096 x 3072 18.4 / 14.3 (K 1536
// 10.9 / 11.3), of more 127 x 4096 x 5504 29.1 / 26.8, x 11008 54.8 / 45.8, 64 x 8192 x 8192 43.7 / 39.4 (127 x 4096 x 4096 21.6 / 21.0); with a second
// round 65 x 4096 x 11008 40.1 / 43.6.  The pair of up to half as many tiles 64 x 4096 x 1536 23.6 / 17.7, two thirds 64 x 5504 x 2752 38.1 / 29.1 (K 1024 16.0 /
// 19.2), more 127 x 4096 x 4096 48.9 / 38.2; with a second round 65 x 2048 x 1536 18.5 / 20.9, 96 x 4096 x 4096 44.7 / 38.3 (K 2048 25 / 27).
static bool narrow_split_is_ahead(const MfmaArgs& a, bool dual) {
  const int64_t t = quad_tiles(a, 1, 2), cu = compute_units();
  if (t > cu || !gemm_rows_apply(a)) return false;
  const bool one_round = (2 * cu + t - 1) / t * t <= 2 * cu + 8, half = t * 2 <= cu;
  if (!dual) return a.K >= (!one_round ? 9216 : (half ? 2048 : 5120));
  return a.K >= (!one_round ? (half ? 1792 : 2432) : (half ? 1024 : (t * 16 <= cu * 11 ? 1280 : 1792)));
}

// The pair of 128 aligned rows and more with a K of 1024 and more: the 64 x 64 tiles of mfma_gemm.hip where these are at most one per compute unit, and the
// 64 x 192 ring of mfma_mid.hip where that takes the shape with hardly a padded column and 64 x 96 would serve it here.  us here / there, weights from HBM:
// 128 x 2752 x 1536 21.8 / 20.1, 256 x 4096 x 2432 31.3 / 28.5 (K 1024 15.4 / 15.1, 768 11.2 / 13.1); 256 x 11008 x 1536 41.1 / 38.8, 575 x 4964 x 1536 39.1 /
// 35.7 (256 x 11008 x 512 16.6 / 17.2, 800 x 2752 x 1536, a twentieth of it padding, 32.1 / 33.5).
static bool pair_of_64_is_ahead(const MfmaArgs& a) {
  if (a.B < 128 || a.K < 1024) return false;
  if (quad_tiles(a, 2, 2) <= compute_units()) return true;
  const int64_t wide = ((int64_t)a.N + 191) / 192 * 192;
  return (int64_t)a.N * 29 >= wide * 28 && quad_pick(a, true, false).form == 8 && gemm_mid_pair_of_64(a);
}

// Ragged rows: the tiles here take up to twice their costs with them (256 x 4096 x 4098 34 us, 18 by the table), so that the register pipelines of mfma_gemm.hip
// and mfma_mid.hip are ahead on few or small tiles.  us here / there, weights from HBM:
//   a pair of up to 127 rows with at most one of the 32 x 64 tiles per compute unit, 64 x 5504 x 746 18.4 / 14.7, 33 x 4096 x 2050 38.6 / 25.8 (65 x 5504 x 746,
//     one and a little, 14.8 / 15.4); of more rows with at most one 64 x 64 tile from a K of 1152 on, 154 x 1376 x 2050 35.9 / 30.8 (128 x 4096 x 1492 31.2 / 31.5);
//   a single matrix with at most one 32 x 64 tile per compute unit, 128 x 4096 x 1492 15.7 / 11.5, 256 x 704 x 2050 18.2 / 12.5 (K 322 as fast); with padded row
//     tiles from a K of 2048 on, or 1000 where they are few (200 x 1002 x 746 6.7 / 7.7, 154 x 256 x 1492 9.9 / 8.5);
//   one that the 64 x 128 ring takes, unless 96 x 64 serves it here, 512 x 4096 x 1492 24.2 / 20.3 (1500 x 704 x 1492 on 96 x 64 15.3 / 18.2); one that the
//     128 x 128 ring takes and 96 x 64 would serve here, of up to 192 rows from 1280 on, 154 x 11008 x 4098 65.6 / 58.0, else from 6144 on;
//   64 x 64 tiles here without padded rows from 1280 on, 256 x 4096 x 4098 34.2 / 28.9, x 1492 15.5 / 14.4 (200 x 4096 x 1492 10.4 / 12.8, x 2050 12.8 / 14.8),
//     with them from 2048 on and more than one per compute unit; 96 x 64 that fill three quarters of the chip with up to 192 rows, 154 x 5504 x 4098 37.5 / 34.3.
static bool ragged_is_ahead_elsewhere(const MfmaArgs& a, bool dual) {
  const int64_t cu = compute_units(), t32 = quad_tiles(a, 1, 2), t64 = quad_tiles(a, 2, 2);
  if (dual) return a.B < 128 ? t32 <= cu : a.K >= 1152 && t64 <= cu;
  const bool full = rows_fill(a);
  if (t32 <= cu) return full || a.K >= 2048 || (t32 * 4 <= cu && a.K >= 1000);
  const int ring = gemm_mid_ragged_rows(a), form = quad_pick(a, false, true).form;
  if (ring == 64) return form != 10;
  if (ring == 128) return form == 10 && a.K >= (a.B <= 192 ? 1280 : 6144);
  if (form == 12) return full ? a.K >= 1280 : a.K >= 2048 && t64 > cu;
  return form == 10 && a.B <= 192 && a.K >= 2048 && quad_tiles(a, 3, 2) * 4 <= 3 * cu;
}

bool gemm_quad_apply(const MfmaArgs& a, bool dual) {
  if (!quad_range(a, dual)) return false;
  if (a.B < 128 && quad_grid(a, dual)) return !narrow_split_is_ahead(a, dual);
  if (quad_grid(a, dual)) return dual ? !pair_of_64_is_ahead(a) : !split_is_ahead(a);
  return quad_words(a, dual) && (dual || a.B >= 128) && !ragged_is_ahead_elsewhere(a, dual);
}

template <int DT>
static int launch_gemm_quad_dt(const MfmaArgs& a, bool dual, hipStream_t st, const char* who) {
  QuadArgs q{};
  q.a[0] = a;
  const bool any = !quad_grid(a, dual);
  if (!dual && !any) {
    const ShareForm f = share_form(a);
    if (f.shares > 0) {
      q.shares = f.shares;
      q.per = f.per;
      q.part = a.scratch;
      q.us = share_us(f.bm, f.bn, quad_tiles(a, f.bm / 32, f.bn / 32) * f.shares, f.per, compute_units());
      return launch_share_dt<DT>(q, f, st, who);
    }
  }
  const QuadSums sums = dual || any ? QuadSums{kOrderPlain, 0} : quad_sums(a);
  const QuadPick pick = quad_pick(a, dual, any, sums.order);
  const int form = pick.form;
  q.us = pick.us;
#define FSVD_QUAD_CASE(EPI, RAG, n, TM, TN, SX, SW, OCC) case n: return launch_quad_t<DT, EPI, TM, TN, SX, SW, OCC, RAG>(q, st, who);
  if (dual && any) {
    switch (form) {
#define X(n, TM, TN, SX, SW, OCC, ...) FSVD_QUAD_CASE(kQuadPair, true, n, TM, TN, SX, SW, OCC)
      FSVD_QUAD_PAIR_ANY(X)
#undef X
    }
  } else if (dual) {
    switch (form) {
#define X(n, TM, TN, SX, SW, OCC, ...) FSVD_QUAD_CASE(kQuadPair, false, n, TM, TN, SX, SW, OCC)
      FSVD_QUAD_PAIR(X)
#undef X
    }
  } else if (any) {
    switch (form) {
#define X(n, TM, TN, SX, SW, OCC, ...) FSVD_QUAD_CASE(kQuadPlain, true, n, TM, TN, SX, SW, OCC)
      FSVD_QUAD_PLAIN_ANY(X)
#undef X
    }
  } else if (sums.order == kOrderCut) {
    q.per = sums.per;
    return launch_quad_t<DT, kQuadPlain, 2, 2, 5, 5, 2, false, 1, true>(q, st, who);
  } else if (sums.order == kOrderHalves) {
    switch (form) {
#define X(n, TM, TN, SX, SW, OCC, ...) case n: if constexpr (quad_halves(n)) return launch_quad_t<DT, kQuadPlain, TM, TN, SX, SW, OCC, false, 2>(q, st, who); break;
      FSVD_QUAD_PLAIN(X)
#undef X
    }
  } else {
    switch (form) {
#define X(n, TM, TN, SX, SW, OCC, ...) FSVD_QUAD_CASE(kQuadPlain, false, n, TM, TN, SX, SW, OCC)
      FSVD_QUAD_PLAIN(X)
#undef X
    }
  }
  set_last_error("%s: no tile for %d x %d x %d", who, a.B, a.N, a.K);
  return kErrBadShape;
}
int launch_gemm_quad(const MfmaArgs& a, bool dual, hipStream_t st, const char* who) {
  return a.dt == 1 ? launch_gemm_quad_dt<1>(a, dual, st, who) : launch_gemm_quad_dt<0>(a, dual, st, who);
}

}  // namespace fsvd
