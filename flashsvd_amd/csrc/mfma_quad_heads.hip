// Head expansions of prompts (q, k and v in one launch, rotation and store fused) on the four-wave tiles of mfma_quad.hpp.
#include "mfma_quad.hpp"

namespace fsvd {

// Tiles and their costs as in mfma_quad.hip, per round and K step in us.  A tile takes whole units of sixteen columns and the sixteen 64 past
// them.  q, k and v of 32 heads at rank 1024 with weights from HBM, 64 x 128 rings and 256 x 256 tiles before -> these: 154 / 333 / 512 / 1024 /
// 2048 / 4096 rows 18.6 -> 15.0, 25.2 -> 20.5, 28.3 -> 25.7, 42.2 -> 39.7, 82.3 -> 70.1, 125.9 -> 115.2; at rank 1664 and 16384 rows 696 -> 594;
// 24 / 64 rows 12.3 -> 9.0, 13.5 -> 10.2.
#define FSVD_QUAD_HEADS(X) \
  X(0, 8, 8, 2, 3, 1, 0.f, 0.f, 15.75f, 1.109f) X(1, 6, 4, 2, 2, 2, 5.73f, 0.855f, 8.07f, 1.176f) X(2, 5, 4, 2, 2, 2, 4.70f, 0.822f, 8.12f, 1.018f) \
  X(3, 4, 4, 2, 3, 2, 4.44f, 0.540f, 6.92f, 0.861f) X(4, 3, 4, 2, 3, 2, 3.30f, 0.512f, 5.36f, 0.715f) X(5, 2, 4, 3, 4, 1, 0.f, 0.f, 3.01f, 0.359f) \
  X(6, 2, 2, 5, 5, 2, 2.39f, 0.196f, 3.13f, 0.394f)
#define FSVD_QUAD_HEADS_ANY(X) X(3, 4, 4, 2, 3, 2) X(4, 3, 4, 2, 3, 2) X(6, 2, 2, 4, 4, 2)

static int heads_pick(const ExpandArgs* d, int n, bool any, float& us_out) {
  const int64_t rows = (int64_t)d[0].B * d[0].M, cu = compute_units();
  int best = -1;
  float best_us = 0.f, steps = 0.f;
  for (int k = 0; k < n; ++k) steps = std::max(steps, (float)((d[k].R + 63) / 64));
  const auto take = [&](int form, int tm, int tn, int occ, const QuadCost& c) {
    int64_t tiles = 0;
    for (int k = 0; k < n; ++k) tiles += ((int64_t)d[k].heads * 128 + 32 * tn - 1) / (32 * tn);
    tiles *= (rows + 32 * tm - 1) / (32 * tm);
    const float us = quad_us(c, tiles, occ, steps, cu);
    if (best < 0 || us < best_us) { best = form; best_us = us; }
  };
#define X(n_, TM, TN, SX, SW, OCC, F1, S1, F2, S2) if (!any || n_ == 3 || n_ == 4 || n_ == 6) take(n_, TM, TN, OCC, QuadCost{F1, S1, F2, S2});
  FSVD_QUAD_HEADS(X)
#undef X
  us_out = best_us;
  return best;
}
static bool heads_on_grid(const ExpandArgs& a) { return a.R % 64 == 0 && a.sp_b % 8 == 0 && a.sp_m % 8 == 0 && a.ldu % 8 == 0 && aligned16(a.p) && aligned16(a.u); }
// the same rank in a launch where it is no whole number of steps (the tail is cleared by one rank)
bool expand_quad_apply(const ExpandArgs* d, int n) {
  if (compute_units() <= 0 || (int64_t)d[0].B * d[0].M < 17) return false;
  bool any = false;
  for (int k = 0; k < n; ++k) any = any || !heads_on_grid(d[k]);
  for (int k = 0; k < n; ++k) {
    const ExpandArgs& a = d[k];
    const auto al4 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3) == 0; };
    if (a.R < 320 || a.sp_b < 0 || a.sp_m < 0 || ((a.B - 1) * a.sp_b + (a.M - 1) * a.sp_m + a.R) * 2 >= (int64_t)4 << 30 || !below_4gib((int64_t)a.heads * 128, a.ldu)) return false;
    if (any && (a.R != d[0].R || a.sp_b % 2 || a.sp_m % 2 || a.ldu % 2 || !al4(a.p) || !al4(a.u))) return false;
  }
  return true;
}
template <int DT>
static int launch_expand_quad_dt(const ExpandArgs* d, int n, hipStream_t st) {
  const char* who = "fsvd_lowrank_expand_heads";
  bool any = false;
  for (int k = 0; k < n; ++k) any = any || !heads_on_grid(d[k]);
  QuadArgs q{};
  const int rows = d[0].B * d[0].M;
  for (int k = 0; k < n; ++k) {
    const ExpandArgs& a = d[k];
    q.a[k] = MfmaArgs{a.p, 0, 0, a.u, nullptr, a.ldu, a.bias, nullptr, 0, a.y, 0, rows, a.heads * 128, a.R, 0};
    q.ep[k] = ExpandEpi{a.cos, a.sin, a.rope_len, a.positions, a.M, a.sp_b, a.sp_m, a.sy_b, a.sy_m, a.sy_h, a.dst_by_position, a.dst_rows, a.pos0};
  }
  const auto tile = [&](int bn) {
    int tiles = 0;
    for (int k = 0; k < 4; ++k) {
      q.first[k] = tiles;
      if (k < n) tiles += (d[k].heads * 128 + bn - 1) / bn;
    }
    q.nt = tiles;
  };
  q.a[0].next = d[0].next;
  const int form = heads_pick(d, n, any, q.us);
  if (any) {
    switch (form) {
#define X(n_, TM, TN, SX, SW, OCC) case n_: tile(32 * TN); return launch_quad_t<DT, kQuadHeads, TM, TN, SX, SW, OCC, true>(q, st, who);
      FSVD_QUAD_HEADS_ANY(X)
#undef X
    }
  } else {
    switch (form) {
#define X(n_, TM, TN, SX, SW, OCC, ...) case n_: tile(32 * TN); return launch_quad_t<DT, kQuadHeads, TM, TN, SX, SW, OCC>(q, st, who);
      FSVD_QUAD_HEADS(X)
#undef X
    }
  }
  set_last_error("%s: no tile for %d rows", who, rows);
  return kErrBadShape;
}
int launch_expand_quad(const ExpandArgs* d, int n, hipStream_t st) {
  return d[0].dt == 1 ? launch_expand_quad_dt<1>(d, n, st) : launch_expand_quad_dt<0>(d, n, st);
}

}  // namespace fsvd
