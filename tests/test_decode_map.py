"""The assignment of a decode attention launch's workgroups (csrc/decode_map.hpp), compiled on the host from the header that the
kernels include: every key range of every head of every sequence has one workgroup."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "flashsvd_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "decode_map.hpp"
using namespace fsvd;
template <class F>
bool every_part(F slot, const char* how, int B, int H, int nsplit) {
  std::vector<int> seen((size_t)B * H * nsplit);
  for (int id = 0; id < B * H * nsplit; ++id) {
    const DecodeSlot t = slot(id, B, H, nsplit);
    if (t.s < 0 || t.s >= nsplit || t.h < 0 || t.h >= H || t.seq < 0 || t.seq >= B || seen[((size_t)t.seq * H + t.h) * nsplit + t.s]++) {
      printf("%d %d %d %s: workgroup %d is outside or takes a part twice\n", B, H, nsplit, how, id);
      return false;
    }
  }
  return true;
}
int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4) {
    const int dh = atoi(argv[i]), B = atoi(argv[i + 1]), H = atoi(argv[i + 2]), nsplit = atoi(argv[i + 3]);
    if (B * H % 8 == 0 && H % 8 == 0 && !every_part(decode_slot_by_length, "by length", B, H, nsplit)) return 1;
    if (!every_part(decode_slot_by_pair, "by pair", B, H, nsplit) || !every_part(decode_slot_by_range, "by range", B, H, nsplit)) return 1;
    for (int hk : {1, 2, H}) {
      if (H % hk) continue;
      for (int group : {1, 2, 4}) {
        if (H / hk % group) continue;
        const DecodePlan p = decode_plan(dh, group, B, H, hk, nsplit);
        const int heads = H / group, same = H / hk / group;
        // by length only what a wave can sort; a kv head on two XCDs only for long sequences without ranges
        if (p.by_length > 0.f && (B < 5 || B > 64 || heads % 8 || (heads / 8 % same && (nsplit > 1 || p.by_length_short > 0.f)))) { printf("%d %d %d %d over %d: by length\n", dh, B, H, nsplit, hk); return 1; }
        // one range each only where that makes full rounds of workgroups
        if (p.one_below && (B * heads < 256 || (B * heads + 255) / 256 * 256 * 9 > B * heads * 10)) { printf("%d %d %d %d over %d: one range\n", dh, B, H, nsplit, hk); return 1; }
        for (int n = 0; n < 5000; n += 1 + n / 50) {
          const int r = decode_ranges(p.one_below, nsplit, n);
          if (r < 1 || r > nsplit || (r > 1 && (r - 1) * 128 >= n)) { printf("%d %d %d %d: %d keys in %d ranges\n", dh, B, H, nsplit, n, r); return 1; }
        }
      }
    }
  }
  return 0;
}
"""


def _build(tmp_path, program):
    src, exe = tmp_path / "map.cpp", tmp_path / "map"
    src.write_text(program)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def test_every_range_has_one_workgroup(tmp_path):
    shapes = [(dh, B, H, nsplit) for dh in (64, 128) for B in (1, 2, 3, 7, 16, 33, 63, 64, 65) for H in (1, 5, 8, 12, 16, 24, 32, 128) for nsplit in (1, 2, 3, 9, 32)]
    r = subprocess.run([str(_build(tmp_path, PROGRAM)), *(str(v) for s in shapes for v in s)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_what_the_shape_decides(tmp_path):
    """The query heads of a kv head stay on one XCD where there are ranges; a second round of workgroups that is nearly empty is no reason for one range."""
    _build(tmp_path, """#include "decode_map.hpp"
using namespace fsvd;
static_assert(decode_plan(128, 1, 48, 16, 2, 2).by_length == 0.f && decode_plan(128, 2, 48, 16, 2, 2).by_length == 0.f);
static_assert(decode_plan(128, 2, 36, 32, 4, 1).by_length == 1.5f && decode_plan(128, 2, 36, 32, 4, 1).by_length_short == 0.f);
static_assert(decode_plan(128, 4, 16, 32, 8, 4).by_length == kDecodeAlways && decode_plan(128, 1, 5, 40, 8, 10).by_length == kDecodeAlways);
static_assert(decode_plan(128, 4, 14, 64, 8, 2).by_length == 1.2f && decode_plan(128, 4, 64, 32, 8, 1).by_length_short == 1.5f);
static_assert(decode_plan(128, 2, 24, 32, 8, 2).by_length_short == 0.f && decode_plan(128, 2, 40, 32, 8, 1).by_length_short == 1.5f);
static_assert(decode_plan(64, 1, 16, 32, 32, 4).by_length == 0.f && decode_plan(128, 1, 4, 32, 32, 4).by_length == 0.f);
static_assert(decode_plan(128, 1, 24, 12, 12, 7).one_below == 0 && decode_plan(64, 1, 24, 12, 12, 7).one_below == 0);
static_assert(decode_plan(128, 1, 16, 32, 32, 4).one_below == 1536 && decode_plan(64, 1, 16, 16, 16, 3).one_below == 512);
static_assert(decode_plan(128, 1, 16, 32, 32, 1).one_below == 0 && decode_plan(128, 4, 64, 32, 8, 2).one_below == 0);
int main() { return 0; }
""")


def test_assignment_of_many_pairs_is_a_constant_expression(tmp_path):
    """131072 (sequence, head) pairs and more: the arithmetic stays within 32 bits (a constant expression that overflows does not
    compile), and the ranges of a pair go an equal share of an XCD's workgroups apart."""
    asserts = []
    for B, H, nsplit in ((4096, 32, 1), (16384, 32, 4), (65536, 33, 2), (1, 1 << 18, 3)):
        per = B * H // (8 if B * H % 8 == 0 else 1)
        for s in range(nsplit):
            first, xcds = s * per, 8 if B * H % 8 == 0 else 1
            pair = s * max(1, per // nsplit) % per
            asserts.append(f"constexpr auto t{len(asserts)} = decode_slot_by_pair({first * xcds}, {B}, {H}, {nsplit});\n"
                           f"constexpr auto r{len(asserts)} = decode_slot_by_range({first}, {B}, {H}, {nsplit});\n"
                           f"constexpr auto p{len(asserts)} = decode_plan(64, 1, {B}, {H}, {H}, {nsplit});\n"
                           f"static_assert(t{len(asserts)}.s == {s} && t{len(asserts)}.h == {pair % H} && t{len(asserts)}.seq == {pair // H});")
    _build(tmp_path, '#include "decode_map.hpp"\nusing namespace fsvd;\n' + "\n".join(asserts) + "\nint main() { return 0; }\n")


def test_one_range_keeps_the_group(tmp_path):
    """Calls over 129 to 256 rows that run as one range keep the query heads together that a workgroup of two ranges takes where these are all heads of a
    kv head, whose new row the launch then appends itself, and with head_dim 64; the group of all other calls goes by their ranges."""
    from flashsvd_amd.hip_ops import pick_nsplit
    asserts = []
    for dh in (64, 128):
        for B in (1, 8, 9, 15, 16, 24, 31, 32, 40, 63, 64, 100):
            for H, hk in ((8, 8), (8, 2), (16, 8), (32, 32), (32, 16), (32, 8), (32, 1), (64, 8), (28, 4), (40, 8)):
                for S in (1, 128, 129, 200, 256, 257):
                    def group(n, rep=H // hk):
                        return 4 if rep % 4 == 0 and B * (H // 4) * n >= 512 else (2 if dh == 128 and rep % 2 == 0 and B * (H // 2) * n >= 512 else 1)
                    ranges, n = max(1, min((S + 127) // 128, max(1, 2048 // (B * H)))), pick_nsplit(S, B, H, dh)
                    for appends in (0, 1):
                        keeps = dh == 64 or (appends and group(ranges) == H // hk)
                        want = group(ranges) if keeps else group(n)
                        asserts.append(f"static_assert(decode_group({dh}, {B}, {H}, {hk}, {S}, {n}, {appends}) == {want});")
                        asserts.append(f"static_assert(decode_group({dh}, {B}, {H}, {hk}, {S}, {ranges}, {appends}) == {group(ranges)});")
    _build(tmp_path, '#include "decode_map.hpp"\nusing namespace fsvd;\n' + "\n".join(asserts) + "\nint main() { return 0; }\n")


def test_one_pass_of_256_keys_takes_few_pairs(tmp_path):
    """More than 1024 pairs have one range whatever the cache's length and stay with passes of 128 keys, as other cache lengths and ranges do."""
    _build(tmp_path, """#include "decode_map.hpp"
using namespace fsvd;
static_assert(decode_one_pass(64, 1, 8, 129, 1) && decode_one_pass(64, 32, 32, 256, 1) && decode_one_pass(64, 1, 1024, 200, 1));
static_assert(!decode_one_pass(64, 33, 32, 256, 1) && !decode_one_pass(64, 64, 32, 137, 1) && !decode_one_pass(64, 65536, 65536, 200, 1));
static_assert(!decode_one_pass(64, 1, 8, 128, 1) && !decode_one_pass(64, 1, 8, 257, 1) && !decode_one_pass(64, 1, 8, 200, 2) && !decode_one_pass(128, 1, 8, 200, 1));
int main() { return 0; }
""")


def test_ranges_of_calls_that_append_rows_of_their_own():
    """head_dim 128 and a kv head per head: with an appended row, a second round of workgroups that is less than five eighths full keeps two ranges."""
    from flashsvd_amd.hip_ops import pick_nsplit
    for batch, heads in ((17, 16), (24, 16), (36, 8), (9, 32), (12, 32), (257, 1), (415, 1)):
        assert pick_nsplit(256, batch, heads, 128, own_row=True) == 2 and pick_nsplit(256, batch, heads, 128) == 1
        assert pick_nsplit(128, batch, heads, 128, own_row=True) == 1 and pick_nsplit(200, batch, heads, 64, own_row=True) == 1
    for batch, heads in ((8, 32), (16, 16), (26, 16), (13, 32), (416, 1), (32, 32), (64, 32)):
        assert pick_nsplit(256, batch, heads, 128, own_row=True) == 1
    for batch, heads in ((1, 32), (7, 32), (255, 1)):
        assert pick_nsplit(256, batch, heads, 128, own_row=True) == pick_nsplit(256, batch, heads, 128) == 2
    for length in (257, 4096):
        assert pick_nsplit(length, 9, 32, 128, own_row=True) == pick_nsplit(length, 9, 32, 128)
