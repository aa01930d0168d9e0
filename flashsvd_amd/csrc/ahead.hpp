// Weights that a launch asks for on behalf of those behind it: which ranges, and by how many workgroups.  Arithmetic without device state, evaluated by the launches
// of capi.hip and mfma_quad.hpp and, on the host, by a test.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace fsvd {

// Weights that the next launch reads, asked for by one that leaves the memory or compute units idle: they then come out of the 256 MB in front of HBM.
struct Ahead { const unsigned char* p = nullptr; uint32_t bytes = 0; };
struct AheadList { Ahead r[3]; };                      // in the order of their use

// The whole 16-byte pieces inside `bytes` bytes from p on: where they start and how many they are.
constexpr uintptr_t ahead_first(uintptr_t p) { return (p + 15) & ~(uintptr_t)15; }
constexpr int ahead_pieces(uintptr_t p, uint32_t bytes) {
  const uintptr_t first = ahead_first(p), end = (p + bytes) & ~(uintptr_t)15;
  return end > first ? (int)((end - first) >> 4) : 0;
}

// Weights [N, K] as a range to ask for ahead of their use: rows that lie (nearly) one behind the other, below 1 GiB.
inline Ahead weights_ahead(const void* W, int64_t ldw, int64_t N, int64_t K) {
  Ahead a;
  const int64_t bytes = ((N - 1) * ldw + K) * 2;
  if (N > 0 && K > 0 && ldw >= K && ldw <= K + K / 8 && bytes < (int64_t)1 << 30) {
    a.p = static_cast<const unsigned char*>(W);
    a.bytes = (uint32_t)bytes;
  }
  return a;
}
// What the RMSNorm in front of a rank projection asks for on its behalf: 240 to 1536 rows that fill their tiles of 64 but for a sixteenth, up to 32 MB
// of weights whose rows lie (nearly) one behind the other.  The tiles there take 7 of 25 us longer with weights from HBM than out of the 256 MB in front
// of it (512 x 3072 x 4096), which deeper stages, or a wave of the workgroup that requests lines 3 to 16 steps ahead, do not change: the loads of a
// compute unit come back in order.  us of a whole MLP (norm, rank projection, pair, down projection), without -> with, all weights from HBM:
//   4096 x 11008 at rank 1536: 240 / 256 / 320 / 448 / 512 / 640 / 768 / 1024 / 1536 rows 95.5 -> 93.7, 97.7 -> 95.0, 101.8 -> 97.5, 117.7 -> 113.3, 128.9 -> 124.9,
//     142.1 -> 138.3, 169.6 -> 161.5, 195.0 -> 192.3, 270.5 -> 267.1; at rank 1024 320 / 512 / 1024 rows 81.3 -> 77.0, 98.1 -> 93.6, 156.6 -> 151.0;
//   2048 x 5504 at rank 1024: 256 / 512 / 1024 rows 52.2 -> 49.7, 67.5 -> 65.6, 91.9 -> 89.1.
// What it leaves out: padded row tiles, which wait less (rank 1536, 257 / 333 / 350 rows 98.0 -> 98.8, 105.5 -> 105.7, 108.4 -> 108.5); fewer rows, where the norm grows by
// what the projection gains (16 / 32 / 208 rows 47.5 -> 49.1, 57.9 -> 59.6, 89.4 -> 90.2); more rows (2048 319.5 -> 326.7); 40 MB (rank 2432, 512 / 1024 rows
// 171.4 -> 166.4, 272 -> 277).
inline Ahead norm_ahead(const void* W, int64_t ldw, int64_t B, int64_t N, int64_t K) {
  const Ahead a = weights_ahead(W, ldw, N, K);
  return B >= 240 && B <= 1536 && B * 16 >= (B + 63) / 64 * 64 * 15 && a.bytes <= 32u << 20 ? a : Ahead{};
}

// Workgroups for the `idle` compute units that a launch of `us` leaves, and what they ask for: the ranges of `next`, in their
// order, that they get through at 46 bytes per ns and compute unit while the launch is expected to last, the padding of its row tiles (`rows` in
// `tile_rows`) counted out (128 x 192 tiles over 400 rows end early: with down_v asked for all the same the MLP at rank 2432 went from 146 to 152 us).  A range in part gains
// nothing, its launch takes as long as its slowest workgroups (ranges cut off at 15, 25, 40 bytes per ns: a prompt of 512 tokens 7027 -> 7014, 7010, 6880 us).
// A compute unit reads about 60 from HBM; more than 46 outlasts some launches (54: rank 1024, 384 rows 83.7 -> 88.4, rank 2432, 512 rows 171 -> 177), less
// takes fewer ranges: 46 / 40 / 34 took 0.968, 0.970, 0.977 of the time without over 114 MLPs of 64 to 768 rows (4096 x 11008 at rank 1024, 1492, 1536, 2432, 2048 x 5504 at 704
// and 1024) and 0.978, 0.980, 0.982 over 65 attention halves of 40 to 1024 rows (rank 512 to 1664, 16 and 32 heads over 8 to 32), weights from HBM.
// us without -> with: the pair 512 x 11008 x 1536 leaves 24 compute units to down_v, whose launches then take 26 instead of 36.  MLPs of 4096 x 11008 at rank 1536, 64 / 128
// / 154 / 256 / 333 / 384 / 400 / 512 / 640 / 700 / 768 rows 81.0 -> 77.8, 75.1 -> 73.1, 79.7 -> 79.0, 94.5 -> 90.3, 106.2 -> 105.7, 113.5 -> 107.9, 110.4 -> 110.3, 125.8 -> 116.9, 138.9 ->
// 131.6, 156.5 -> 151.8, 166.5 -> 158.7, at rank 1492 384 / 768 rows 133.5 -> 126.2, 214.3 -> 191.1, 2048 x 5504 at rank 1024 192 / 300 / 400 / 700 rows 54.3 -> 48.2, 56.9 -> 51.9, 64.5 ->
// 64.3, 78.8 -> 71.9; attention halves of 32 heads at rank 1024, 128 / 256 / 333 / 512 rows 56.8 -> 55.7, 67.2 -> 64.3, 81.5 -> 80.9, 93.5 -> 93.6, at rank 1664 512 rows 126.7 -> 119.0.
// What loses: an MLP at rank 2432, 200 rows 117.2 -> 118.7, 2048 x 5504 at rank 1024, 64 rows 48.0 -> 48.4, attention of 32 heads at rank 1024, 200 rows 62.4 -> 62.8, at
// rank 704, 700 rows 103.4 -> 105.0; the others are within 0.7 % of it or ahead.  Launches whose tiles walk K in ranges (ranges_us in quad_costs.hpp) are the idlest: MLPs of 3072 x
// 8192 at rank 1152 / 704 / 512, 192 / 320 / 320 rows, whose rank projection asks for nothing -> asks as well, 63.7 -> 60.0, 57.6 -> 54.9, 51.1 -> 49.3.
// More tiles than compute units: nobody is idle, nothing is asked for.
constexpr float kAheadRate = 46.f;
struct AheadChoice { AheadList ranges; int workgroups; };
inline AheadChoice ahead_choice(const AheadList* next, float us, int64_t rows, int64_t tile_rows, int64_t idle) {
  AheadChoice c{AheadList{}, 0};
  if (next == nullptr || idle <= 0) return c;
  const int64_t room = (int64_t)(us * kAheadRate * 1000.f * (float)rows / (float)tile_rows) * idle;
  int64_t sum = 0;
  for (int i = 0; i < 3; ++i) {
    if (sum + next->r[i].bytes > room) break;
    c.ranges.r[i] = next->r[i];
    sum += next->r[i].bytes;
  }
  c.workgroups = (int)std::min<int64_t>(idle, (sum + 32767) / 32768);
  return c;
}

}  // namespace fsvd
