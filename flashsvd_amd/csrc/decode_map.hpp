// Which part of a decode attention call a workgroup takes, and into how many key ranges a sequence is cut: index arithmetic
// without device state, evaluated by the kernels of attn_decode.hip and, on the host, by a test over all workgroups of a launch.
#pragma once

namespace fsvd {

// Key range s of query head (or head group) h of a sequence: the sequence itself, or, by length, its place among the sequences of
// the batch, longest first (equal lengths in their order).
struct DecodeSlot { int s, h, seq; };

// What a call's shape leaves open until the lengths are known in the kernel.
constexpr int kDecodeLong = 1000, kDecodeShort = 257;
constexpr float kDecodeAlways = 1.f;
struct DecodePlan {
  int one_below;       // sequences of fewer keys run in one range (0: none does)
  int one_if_even;     // ... only while the longest is at most 1.5 times the mean
  float by_length, by_length_short;     // sequences by length where the longest exceeds this many times the mean (0: never); from kDecodeLong, kDecodeShort keys on
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
// keys of 32 heads 68 in that order, 71 by length).  An XCD takes some heads of every sequence instead of every head of some.
//   A sequence of kDecodeLong keys and more: always, the reversed rounds and the eight XCDs share what there is more evenly even where
//     all are alike (16 x 3000 to 4001 keys of 32 heads over 8 51.0 -> 49.0, 33 x up to 4001 128 -> 78, 8 x 4001 over 16 58 -> 47, 5 x 2000 to 4001 of 40
//     heads over 8 46 -> 39); with one kv head of an XCD and a last round that is not full only where the longest is 1.2 times the
//     mean (14 x 4001 keys of 64 heads over 8 96 -> 109).
//   Shorter ones, from three passes of keys on (60 x up to 150 keys 13.1 -> 18.6): where the longest is 1.5 times the mean (40 x up to
//     900 keys of 32 heads over 8 33.8 -> 25.7, but 48 x 375 to 500, two heads a group, 28.0 -> 30.4), in groups not over a full odd number of rounds,
//     since every other one runs backwards (24 x up to 900 keys in three 24.1 -> 26.9), without groups with four kv heads of an XCD (1 KB of a
//     row) or 512 pairs (64 x up to 1000 33.1 -> 32.0, 32 x up to 600 with fewer 13.9 -> 15.4).
//   The query heads of a kv head on different XCDs read it twice (eight over one: 48 x 500 keys 18.7 -> 27.1, 48 x up to 2500 in two ranges
//     37 -> 56): only long and uneven ones for which there are no ranges (36 x up to 1500 keys of 32 heads over 4 46 -> 33).
// With head_dim 64 the pieces are too short (64 x 1000 keys 98.7 -> 105), and up to four sequences leave nothing to sort.
constexpr DecodePlan decode_plan(int head_dim, int group, int B, int H, int Hk, int nsplit) {
  const int heads = H / group, same_kv = H / Hk / group;
  const long pairs = (long)B * heads, rounds = (pairs + 255) / 256, all_rounds = (pairs * nsplit + 255) / 256;
  DecodePlan p{0, 0, 0.f, 0.f};
  if (group == 1 && nsplit > 1 && pairs >= 256 && pairs * 10 >= rounds * 256 * 9 && pairs <= 1 << 20) {
    const int full = 2 * head_dim / 64 * (int)pairs, most = 12 * head_dim;
    p.one_below = full < most ? full : most;
    p.one_if_even = head_dim == 128 && pairs < 512;
  }
  if (head_dim == 128 && heads % 8 == 0 && B > 4 && B <= 64 && pairs <= 1024) {
    const int kv_heads = heads / 8 % same_kv == 0 ? heads / 8 / same_kv : 0;           // of an XCD
    const bool full = pairs * nsplit * 10 >= all_rounds * 256 * 9;
    p.by_length = kv_heads == 0 ? (nsplit == 1 ? 1.5f : 0.f) : (full || kv_heads >= 2 ? kDecodeAlways : 1.2f);
    if (kv_heads > 0 && (group > 1 ? !full || all_rounds % 2 == 0 : kv_heads >= 4 || pairs >= 512)) p.by_length_short = 1.5f;
  }
  return p;
}

// Query heads of a kv head that one workgroup takes: four (head_dim 128: four or two) where the workgroups then still are two per compute unit; groups read
// the rows once and, where they are all heads of the kv head, append the new one themselves.  A cache of 129 to 256 rows and up to 1024 (sequence, head) pairs that
// runs as one range counts as the two that there would be room for, with head_dim 64 and where the call appends (`appends`) and the group keeps that in the launch.
// us at 137 / 248 keys, two ranges with the group, one range without, this; with an append 32 x 32 heads over 8 of 64 10.0, 10.8, 8.6 / 11.4, 13.1, 8.8, of 128
// 13.5, 13.2, 12.4 / 15.5, 14.4, 13.0, 16 x 32 over 16 of 128 10.3, 11.9, 9.3 / 12.2, 13.8, 9.8, none appended 32 x 32 over 8 of 64 9.2, 8.3, 7.8 / 11.1, 10.4, 8.0.
// Elsewhere smaller groups fill the chip better with one range: of 128 and none appended 32 x 32 over 8 12.9, 11.1, 11.5 / 14.9, 11.7, 12.2, 24 x 32 over 16 12.5, 11.3,
// 12.1 / 15.3, 14.4, 13.5; 40 x 32 over 8 of 128, which has one range in any case, 13.9 in twos, 16.2 in fours.
constexpr int decode_group_of(int head_dim, long pairs, int rep, int ranges) {
  if (rep % 4 == 0 && pairs / 4 * ranges >= 512) return 4;
  return head_dim == 128 && rep % 2 == 0 && pairs / 2 * ranges >= 512 ? 2 : 1;
}
constexpr int decode_group(int head_dim, int B, int H, int Hk, int S, int nsplit, bool appends) {
  const int rep = H / Hk;
  const long pairs = (long)B * H;
  if (nsplit == 1 && S > 128 && S <= 256 && pairs <= 1024) {
    const int two = decode_group_of(head_dim, pairs, rep, 2);
    if (head_dim == 64 || (appends && two == rep)) return two;
  }
  return decode_group_of(head_dim, pairs, rep, nsplit);
}

// One range of 129 to 256 rows of 64, one head per workgroup: 256 keys in flight instead of two passes of 128, or two workgroups that meet again in a merge.
// us in two ranges of one pass / one range of two passes / this, 137 and 248 keys: 8 heads 5.6, 4.7, 4.4 and 5.7, 5.1, 5.2; 4 x 32 heads 6.2, 5.4, 5.1 and 6.6, 5.8,
// 5.8; 32 x 16 8.2, 8.0, 7.4 and 10.1, 10.1, 10.2.  Not for more than 1024 (sequence, head) pairs, which had one range before: two passes need half the registers
// and sequences of one pass are ahead there, uneven ones of up to 137 keys, two passes / this: 56 x 32 heads over 4 7.7, 10.1, 64 x 32 13.1, 14.5.
constexpr bool decode_one_pass(int head_dim, int B, int H, int S, int nsplit) {
  return head_dim == 64 && nsplit == 1 && S > 128 && S <= 256 && (long)B * H <= 1024;
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
  const unsigned per = (unsigned)(B * H) >> 3, heads = (unsigned)H >> 3;
  unsigned id = (unsigned)block >> 3;
  if ((id & 32) && (id | 31) < per * nsplit) id ^= 31;
  const unsigned s = id / per, at = id - s * per, seq = at / heads;
  return DecodeSlot{(int)s, (int)((block & 7) * heads + at - seq * heads), (int)seq};
}

// The first range of all heads of an XCD before the second of any, where half of the ranges and more have no keys: those workgroups, which
// leave at once, are the last ones (between the others they left the compute units unevenly loaded: 16 x 1000 keys in one range 93 us).
constexpr DecodeSlot decode_slot_by_pair(int block, int B, int H, int nsplit) {
  const unsigned pairs = B * H;
  const bool by_xcd = (pairs & 7) == 0;
  const unsigned per = by_xcd ? pairs >> 3 : pairs, xcd = by_xcd ? block & 7 : 0, id = by_xcd ? block >> 3 : block;
  const unsigned s = id / per, share = per / (unsigned)nsplit, turn = share > 1 ? share : 1;     // a range later: another compute unit
  const unsigned pair = xcd * per + (id - s * per + s * turn) % per, seq = pair / (unsigned)H;
  return DecodeSlot{(int)s, (int)(pair - seq * H), (int)seq};
}

// The ranges of a head side by side, where most of them have keys (first ranges first: 5 x 2000 keys of 8 heads 13.1 -> 14.0 us, 8 x up to
// 500 of 16 heads of 64 8.0 -> 8.5).
constexpr DecodeSlot decode_slot_by_range(int block, int B, int H, int nsplit) {
  const unsigned total = (unsigned)(B * H) * nsplit, id = (total & 7) == 0 ? (block & 7) * (total >> 3) + ((unsigned)block >> 3) : block;
  const unsigned pair = id / (unsigned)nsplit, seq = pair / (unsigned)H;
  return DecodeSlot{(int)(id - pair * nsplit), (int)(pair - seq * H), (int)seq};
}

}  // namespace fsvd
