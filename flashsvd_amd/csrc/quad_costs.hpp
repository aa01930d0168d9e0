// What the four-wave tiles of mfma_quad.hpp cost: plain arithmetic, evaluated by the launches of mfma_quad.hip and mfma_quad_heads.hip and, on the host, by a
// test of what their launches ask for ahead of its use.
#pragma once
#include <stdint.h>

namespace fsvd {

// What a round of workgroups costs in a form, us: f + s per K step of 64; 1: the compute units hold one workgroup each (or fewer), 2: as many
// as fit.  Fitted to launches with weights from HBM (more of them in turn than the 256 MB in front of it hold) over 125 / 49 / 39 shapes
// (154 to 16384 rows; 1024 to 4096 columns at K 768 to 4096; the pair 5504 x 768 to 11008 x 2432; 48 and 96 heads at rank 512 and 1024):
// the form that they name is on average 2 / 1 / 1 % (at worst 20, 12, 8 %) behind the best of about 30 tilings.  The largest launches take longer than
// they say, whatever the tile (the pair 16384 x 11008 x 2432 1605 us, 1426 by them).
struct QuadCost { float f1, s1, f2, s2; };
constexpr float quad_us(const QuadCost& c, int64_t tiles, int occ, float steps, int64_t cu) {
  const int64_t full = tiles / (cu * occ), rest = tiles - full * cu * occ;
  const float last = rest <= 0 ? 0.f : (occ == 2 && rest <= cu ? c.f1 + c.s1 * steps : c.f2 + c.s2 * steps);
  return (float)full * (c.f2 + c.s2 * steps) + last;
}

//     form, TM, TN, stages of x and W, workgroups per compute unit, costs
#define FSVD_QUAD_PLAIN(X) \
  X(0, 8, 8, 2, 3, 1, 0.f, 0.f, 11.21f, 0.952f) X(1, 8, 6, 2, 3, 1, 0.f, 0.f, 8.57f, 0.783f) X(2, 4, 6, 3, 4, 1, 0.f, 0.f, 4.35f, 0.578f) \
  X(3, 8, 4, 2, 3, 1, 0.f, 0.f, 5.97f, 0.643f) X(4, 6, 4, 3, 4, 1, 0.f, 0.f, 4.84f, 0.502f) X(5, 4, 4, 2, 3, 2, 1.53f, 0.533f, 8.67f, 0.679f) \
  X(6, 4, 4, 4, 5, 1, 0.f, 0.f, 3.03f, 0.450f) X(7, 4, 3, 5, 6, 1, 0.f, 0.f, 4.29f, 0.353f) X(8, 4, 2, 3, 4, 2, 0.57f, 0.339f, 3.94f, 0.568f) \
  X(9, 2, 4, 3, 4, 1, 0.f, 0.f, 1.24f, 0.354f) X(10, 3, 2, 3, 4, 2, 0.24f, 0.297f, 3.14f, 0.440f) X(11, 2, 3, 3, 4, 2, 0.30f, 0.311f, 1.99f, 0.484f) \
  X(12, 2, 2, 5, 5, 2, 0.49f, 0.227f, 2.66f, 0.355f)
constexpr bool quad_halves(int n) { return n >= 8 && n != 9; }      // the forms that shapes with K halved get, with registers for a second set of accumulators
constexpr QuadCost kPlainCosts[] = {
#define X(n, TM, TN, SX, SW, OCC, F1, S1, F2, S2) QuadCost{F1, S1, F2, S2},
  FSVD_QUAD_PLAIN(X)
#undef X
};
constexpr QuadCost kCost256x128Shares{0.f, 0.f, 6.65f, 0.634f};     // three stages of both operands, in shares only
// A launch of `wgs` workgroups that take `per` K steps of a tile each, in shares; tiles of 64 x 64 fit twice on a compute unit and then, as elsewhere, take f1 and s1
// where there are no more of them than compute units (16 steps 4.1 us, and 8.3 for two of them).
constexpr const QuadCost& share_cost(int bm, int bn) {
  return bn == 64 ? kPlainCosts[12] : (bm == 64 ? kPlainCosts[9] : (bm == 128 ? kPlainCosts[6] : kCost256x128Shares));
}
constexpr float share_us(int bm, int bn, int64_t wgs, int per, int64_t cu) { return quad_us(share_cost(bm, bn), wgs, bn == 64 ? 2 : 1, (float)per, cu); }
// The same tiles with K in ranges one after the other (kOrderCut of mfma_quad.hip): the walk of one tile, whatever the ranges.
constexpr float ranges_us(int64_t tiles, int K, int64_t cu) { return quad_us(kPlainCosts[12], tiles, 2, (float)((K + 63) / 64), cu); }

}  // namespace fsvd
