// Which part of a decode attention call a workgroup takes, and into how many key ranges a sequence is cut: index arithmetic
// without device state, evaluated by the kernels of attn_decode.hip and, on the host, by a test over all workgroups of a launch.
#pragma once

namespace fsvd {

// Key range s of query head (or head group) h of a sequence: the sequence itself, or, by length, its place among the sequences of
// the batch, longest first (equal lengths in their order).
struct DecodeSlot { int s, h, seq; };

// Workgroup `block` of B * H * nsplit; H counts the head groups where a workgroup takes a group.
// Consecutive workgroup ids go round-robin over the 8 XCDs: the ranges of one head (which meet again in the merge) run on the same
// XCD, the first range of all its heads before the second of any, so that workgroups without a range, which leave at once, are the
// last ones (between the others they left the compute units unevenly loaded: 16 x 1000 keys 93 us).
// By length: up to 64 sequences with head_dim 128, 1024 pairs (four per compute unit; beyond, the order of dispatch evens things out,
// and 48 x 500 keys of 32 heads are 68 us this way, 71 the other): an XCD takes some heads of every sequence, not every head of some,
// the sequences longest first, and every other 32 workgroups of an XCD (one per compute unit) in reverse, so that the ranges of a
// long and of a short sequence share a compute unit.  Without -> with, 32 heads: 16 x 1 to 1000 keys 31.4 -> 27.0 us, 32 x 1 to
// 1000 55.6 -> 46.2, 16 x 4000 175.6 -> 171.2; 64 x 1 to 1000, four heads a group, 42.7 -> 32.8.  With head_dim 64 the pieces of
// a row that an XCD then reads are too small (64 x 1000 keys 98.7 -> 105).
constexpr bool decode_by_length(int head_dim, int B, int H) { return head_dim == 128 && H % 8 == 0 && B <= 64 && B * H <= 1024; }

// (pairs that are a multiple of 8, as H is)
constexpr DecodeSlot decode_slot_by_length(int block, int B, int H, int nsplit) {
  const int per = (B * H) >> 3, heads = H >> 3;
  int id = block >> 3;
  if ((id & 32) && (id | 31) < per * nsplit) id ^= 31;
  const int s = id / per;
  id -= s * per;
  return DecodeSlot{s, (block & 7) * heads + id % heads, id / heads};
}

constexpr DecodeSlot decode_slot_by_pair(int block, int B, int H, int nsplit) {
  const int pairs = B * H;
  const bool by_xcd = (pairs & 7) == 0;
  const int per = by_xcd ? pairs >> 3 : pairs, xcd = by_xcd ? block & 7 : 0, id = by_xcd ? block >> 3 : block;
  const int s = id / per, share = per / nsplit, turn = share > 1 ? share : 1;     // a range later: another compute unit
  const int pair = xcd * per + (id - s * per + s * turn) % per;
  return DecodeSlot{s, pair % H, pair / H};
}

// Key ranges that a sequence of n keys is cut into, at most nsplit (what the scratch holds): known from the length alone, so
// the same launch serves a cache that is nearly empty and one that is full; the other workgroups of (b, h) leave at once.
// A range holds at least one pass of 128 keys.  Where the heads of all sequences fill the chip by themselves (one query head per
// workgroup, 256 pairs and more) ranges only even out sequences of different lengths: from 2 keys a pair on (one with head_dim 64,
// whose sequences stay on one XCD), and an odd count (the starts of two or four equal ranges lie a power of two apart, and
// their workgroups ask the same memory channels at the same time).  Both sides with 32 heads: 16 x 1000 keys 55.1 us in four
// ranges, 46.9 in one (in a cache of 1024 rows 67.2, 48.9), 32 x 1000 95.6 and 88.4, 16 x 750 to 1000 47.7 and 42.7; one sequence
// of 300 keys in a cache of 4096 rows 13.0 in 32, 6.6 in three.
constexpr int decode_ranges(int head_dim, int group, int B, int H, int nsplit, int n_keys) {
  int n = (n_keys + 127) >> 7;
  n = n < nsplit ? n : nsplit;
  if (group == 1 && B * H >= 256) {
    const int odd = (n_keys / (head_dim / 64 * B * H)) | 1;
    n = n < odd ? n : odd;
  }
  return n > 1 ? n : 1;
}

}  // namespace fsvd
