// Which part of a decode attention call a workgroup takes, and into how many key ranges a sequence is cut: index arithmetic
// without device state, evaluated by the kernels of attn_decode.hip and, on the host, by a test over all workgroups of a launch.
#pragma once

namespace fsvd {

// Key range s of query head (or head group) h of a sequence: the sequence itself, or, by length, its place among the sequences of
// the batch, longest first (equal lengths in their order).
struct DecodeSlot { int s, h, seq; };

// What a call's shape leaves open until the lengths are known in the kernel.
constexpr float kDecodeLong = 1000.f;
struct DecodePlan {
  int one_below;       // sequences of fewer keys run in one range (0: none does)
  int one_if_even;     // ... only while the longest is at most 1.5 times the mean
  float by_length, by_length_short;     // sequences by length where the longest exceeds this many times the mean (0: never); below kDecodeLong keys
};

// B sequences, H query heads over Hk, `group` heads per workgroup, at most nsplit ranges; a pair is a (sequence, group).  Measured per
// call over caches from HBM, us: every key range that there is scratch for -> what is chosen here.
// One range: where the pairs fill the chip by themselves, with one query head per workgroup, 256 pairs and more in rounds that are at
// least 90 percent full (288 pairs of 24 x 900 keys: one range 36.9, seven 31), all sequences below 4 keys a pair (2 with head_dim 64) and 1536
// (768); longer ones lose nothing by ranges (32 x 2000 keys of 16 heads 91.5, in one range 96.5; 16 x 4000 keys of 16 heads of 64 in eight
// ranges 52.7, in eight that start elsewhere 54.6).  Starts of equal ranges lie a power of two apart and their workgroups ask the same memory
// channels at the same time: 16 x 1000 keys of 32 heads 55.1 -> 46.9, 16 x 300 of 16 heads of 64 10.2 -> 8.7.  A single round of fewer
// than 512 pairs of uneven sequences has nothing that evens it out (16 x up to 1000 keys of 16 heads in one range 23.3, in ranges 20.4).
// By length: head_dim 128, up to 64 sequences and 1024 pairs (four per compute unit; beyond, the order of dispatch evens things out: 48 x 500
// keys of 32 heads 68 in that order, 71 by length).  An XCD takes some heads of every sequence instead of every head of some, so the query heads of
// a kv head have to stay together (eight heads over one kv head apart: 48 x 500 keys 18.7 -> 27.1), and its pieces of a row get short: with
// four kv heads of an XCD (1 KB) it pays for long sequences that differ at all (16 x 750 to 1000 keys 47.0 -> 44.4, but 12 x 375 to 500 22.6 ->
// 23.8), with fewer where the longest is 1.5 times the mean (64 x 1 to 1000 keys of four heads a group 45.7 -> 36.0, but 48 x 375 to 500,
// two heads a group, 28.0 -> 30.4, and 64 x 125, 15.0 -> 17.7).  Groups: an even number of rounds, since every other one runs backwards
// (24 x up to 900 keys in three 24.1 -> 26.9).  No groups and two kv heads of an XCD: long ones (5 x up to 2000 keys 16.1 -> 12.8,
// 6 x up to 900 11.4 -> 12.0) or 512 pairs, one: 512 pairs (64 x up to 1000 33.1 -> 32.0, 32 x up to 600 13.9 -> 15.4).  With head_dim 64 the
// pieces are too short (64 x 1000 keys 98.7 -> 105), and up to four sequences leave nothing to sort.
constexpr DecodePlan decode_plan(int head_dim, int group, int B, int H, int Hk, int nsplit) {
  const int heads = H / group, same_kv = H / Hk / group;
  const long pairs = (long)B * heads, rounds = (pairs + 255) / 256, all_rounds = (pairs * nsplit + 255) / 256;
  DecodePlan p{0, 0, 0.f, 0.f};
  if (group == 1 && nsplit > 1 && pairs >= 256 && pairs * 10 >= rounds * 256 * 9 && pairs <= 1 << 20) {
    const int full = 2 * head_dim / 64 * (int)pairs, most = 12 * head_dim;
    p.one_below = full < most ? full : most;
    p.one_if_even = head_dim == 128 && pairs < 512;
  }
  if (head_dim == 128 && heads % 8 == 0 && B > 4 && B <= 64 && pairs <= 1024 && heads / 8 % same_kv == 0) {
    const int kv_heads = heads / 8 / same_kv;           // of an XCD
    if (group > 1 ? all_rounds % 2 == 0 : (kv_heads >= 2 || pairs >= 512)) {
      const bool wide = group == 1 && kv_heads >= 4;
      p.by_length = wide ? 1.05f : 1.5f;
      p.by_length_short = group > 1 || wide || pairs >= 512 ? 1.5f : 0.f;
    }
  }
  return p;
}

// Key ranges that a sequence of n keys is cut into, at most nsplit (what the scratch holds): known from the length alone, so
// the same launch serves a cache that is nearly empty and one that is full; the other workgroups of (b, h) leave at once.
// A range holds at least one pass of 128 keys: one sequence of 300 keys in a cache of 4096 rows 13.0 us in 32 ranges, 6.6 in three.
constexpr int decode_ranges(int one_below, int nsplit, int n_keys) {
  const int n = (n_keys + 127) >> 7, most = n < nsplit ? n : nsplit;
  return n_keys < one_below || most < 1 ? 1 : most;
}

// The three assignments of workgroup `block` of B * H * nsplit; H counts the head groups where a workgroup takes a group.  Consecutive
// workgroup ids go round-robin over the 8 XCDs: the ranges of one head (which meet again in the merge) run on the same XCD.
// By length: an XCD takes some heads of every sequence, the sequences longest first, and every other 32 workgroups of an XCD (one per
// compute unit) in reverse, so that the ranges of a long and of a short sequence share a compute unit (pairs that are a multiple of 8, as H is).
constexpr DecodeSlot decode_slot_by_length(int block, int B, int H, int nsplit) {
  const int per = (B * H) >> 3, heads = H >> 3;
  int id = block >> 3;
  if ((id & 32) && (id | 31) < per * nsplit) id ^= 31;
  const int s = id / per;
  id -= s * per;
  return DecodeSlot{s, (block & 7) * heads + id % heads, id / heads};
}

// The first range of all heads of an XCD before the second of any, where half of the ranges and more have no keys: those workgroups, which
// leave at once, are the last ones (between the others they left the compute units unevenly loaded: 16 x 1000 keys in one range 93 us).
constexpr DecodeSlot decode_slot_by_pair(int block, int B, int H, int nsplit) {
  const int pairs = B * H;
  const bool by_xcd = (pairs & 7) == 0;
  const int per = by_xcd ? pairs >> 3 : pairs, xcd = by_xcd ? block & 7 : 0, id = by_xcd ? block >> 3 : block;
  const int s = id / per, share = per / nsplit, turn = share > 1 ? share : 1;     // a range later: another compute unit
  const int pair = xcd * per + (id - s * per + s * turn) % per;
  return DecodeSlot{s, pair % H, pair / H};
}

// The ranges of a head side by side, where most of them have keys (first ranges first: 5 x 2000 keys of 8 heads 13.1 -> 14.0 us, 8 x up to
// 500 of 16 heads of 64 8.0 -> 8.5).
constexpr DecodeSlot decode_slot_by_range(int block, int B, int H, int nsplit) {
  const int total = B * H * nsplit, id = (total & 7) == 0 ? (block & 7) * (total >> 3) + (block >> 3) : block;
  const int pair = id / nsplit;
  return DecodeSlot{id - pair * nsplit, pair % H, pair / H};
}

}  // namespace fsvd
