"""What a launch asks for ahead of its use (csrc/ahead.hpp), compiled on the host from the header that the launches include: which weights count as a range,
which of them a launch takes and with how many workgroups, and that these read whole pieces inside the range, each at least once."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "flashsvd_amd" / "csrc"

HEAD = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "ahead.hpp"
#include "quad_costs.hpp"
using namespace fsvd;
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); exit(1); } } while (0)
static const void* at(uintptr_t p) { return reinterpret_cast<const void*>(p); }
static bool none(const Ahead& a) { return a.p == nullptr && a.bytes == 0; }
static AheadList list(uint32_t a, uint32_t b, uint32_t c) {
  const unsigned char* p = static_cast<const unsigned char*>(at(4096));
  return AheadList{{Ahead{p, a}, Ahead{p, b}, Ahead{p, c}}};
}
"""


def _run(tmp_path, body):
    src, exe = tmp_path / "ahead.cpp", tmp_path / "ahead"
    src.write_text(HEAD + "int main() {\n" + body + "\n  return 0;\n}\n")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-Wno-unused-function", f"-I{CSRC}", str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_pieces_lie_inside_the_range_and_are_all_read(tmp_path):
    _run(tmp_path, r"""
  for (uintptr_t p = 64; p < 96; ++p)
    for (uint32_t bytes = 0; bytes < 100; ++bytes) {
      int n = 0;
      uintptr_t first = 0;
      for (uintptr_t q = 0; q + 16 <= p + bytes; q += 16)
        if (q >= p && n++ == 0) first = q;
      CHECK(ahead_pieces(p, bytes) == n);
      if (n) CHECK(ahead_first(p) == first);
    }
  CHECK(ahead_pieces(0, 0) == 0 && ahead_pieces(6, (1u << 30) - 2) == (1 << 26) - 1);
  // the loop of request_ahead: eight pieces per thread and turn, clamped to the last one
  for (int threads : {64, 256})
    for (int parts : {1, 3, 190})
      for (int n : {0, 1, 7, 2047, 2048, 2049, 100000}) {
        std::vector<int> seen(n + 1);
        for (int part = 0; part < parts; ++part)
          for (int tid = 0; tid < threads; ++tid)
            for (int i = part * threads * 8 + tid; i < n; i += parts * threads * 8)
              for (int u = 0; u < 8; ++u) seen[std::min(i + u * threads, n - 1)]++;
        for (int i = 0; i < n; ++i) CHECK(seen[i] > 0);
        CHECK(seen[n] == 0);
      }
""")


def test_weights_that_count_as_a_range(tmp_path):
    _run(tmp_path, r"""
  const void* w = at(1000);
  CHECK(weights_ahead(w, 64, 3, 64).bytes == 3 * 128 && weights_ahead(w, 72, 3, 64).bytes == (2 * 72 + 64) * 2 && weights_ahead(w, 64, 3, 64).p == w);
  CHECK(none(weights_ahead(w, 73, 3, 64)) && none(weights_ahead(w, 63, 3, 64)) && none(weights_ahead(w, 0, 3, 64)) && none(weights_ahead(w, -64, 3, 64)));
  CHECK(none(weights_ahead(w, 64, 0, 64)) && none(weights_ahead(w, 64, -5, 64)) && none(weights_ahead(w, 64, 3, 0)));
  CHECK(none(weights_ahead(w, 8192, 65536, 8192)) && weights_ahead(w, 8192, 65535, 8192).bytes == (1u << 30) - 16384);
  // in front of a rank projection: 240 to 1536 rows, their tiles of 64 full but for a sixteenth, up to 32 MB
  for (int rows : {240, 256, 300, 320, 512, 1536}) CHECK(norm_ahead(w, 4096, rows, 4096, 4096).bytes == 32u << 20);
  for (int rows : {1, 64, 192, 239, 257, 299, 333, 1537, 2048}) CHECK(none(norm_ahead(w, 4096, rows, 4096, 4096)));
  CHECK(none(norm_ahead(w, 4096, 512, 4097, 4096)) && none(norm_ahead(w, 5000, 512, 64, 4096)));
""")


def test_whole_ranges_that_fit_into_the_launch(tmp_path):
    """46 bytes per ns and idle compute unit while the launch lasts, padded rows counted out; one workgroup per 32 KB, no more than there are idle units."""
    _run(tmp_path, r"""
  const AheadList l = list(400000, 60000, 1);
  const auto took = [](const AheadChoice& c) { return (c.ranges.r[0].bytes ? 1 : 0) + (c.ranges.r[1].bytes ? 2 : 0) + (c.ranges.r[2].bytes ? 4 : 0); };
  CHECK(took(ahead_choice(nullptr, 10.f, 64, 64, 10)) == 0 && ahead_choice(nullptr, 10.f, 64, 64, 10).workgroups == 0);
  for (int64_t idle : {0, -3}) CHECK(took(ahead_choice(&l, 10.f, 64, 64, idle)) == 0 && ahead_choice(&l, 10.f, 64, 64, idle).workgroups == 0);
  CHECK(ahead_choice(&l, 0.f, 64, 64, 190).workgroups == 0);
  CHECK(took(ahead_choice(&l, 10.f, 64, 64, 1)) == 3 && took(ahead_choice(&l, 10.01f, 64, 64, 1)) == 7);      // 460000 bytes are 10 us of one unit
  CHECK(took(ahead_choice(&l, 9.99f, 64, 64, 1)) == 1 && took(ahead_choice(&l, 8.f, 64, 64, 1)) == 0);         // none behind one that does not fit
  CHECK(took(ahead_choice(&l, 10.f, 48, 64, 1)) == 0 && took(ahead_choice(&l, 10.f, 60, 64, 1)) == 1 && took(ahead_choice(&l, 20.f, 33, 64, 1)) == 7);
  CHECK(ahead_choice(&l, 10.f, 64, 64, 1).workgroups == 1 && ahead_choice(&l, 10.f, 64, 64, 7).workgroups == 7 && ahead_choice(&l, 10.f, 64, 64, 190).workgroups == 15);
  const AheadList hole = list(0, 32768, 32769);
  CHECK(ahead_choice(&hole, 10.f, 64, 64, 190).workgroups == 3 && took(ahead_choice(&hole, 10.f, 64, 64, 190)) == 6);
""")


def test_time_of_a_launch_in_shares(tmp_path):
    """Tiles of 64 x 64 take the time of one per compute unit where there are no more of them; the other tiles are one per compute unit in any case."""
    _run(tmp_path, r"""
  CHECK(share_us(64, 64, 200, 16, 256) == kPlainCosts[12].f1 + kPlainCosts[12].s1 * 16 && share_us(64, 64, 256, 16, 256) == share_us(64, 64, 1, 16, 256));
  CHECK(share_us(64, 64, 257, 16, 256) == kPlainCosts[12].f2 + kPlainCosts[12].s2 * 16 && share_us(64, 64, 512, 16, 256) == share_us(64, 64, 257, 16, 256));
  for (int wgs : {1, 200, 256}) {
    CHECK(share_us(64, 128, wgs, 12, 256) == kPlainCosts[9].f2 + kPlainCosts[9].s2 * 12 && share_us(128, 128, wgs, 12, 256) == kPlainCosts[6].f2 + kPlainCosts[6].s2 * 12);
    CHECK(share_us(256, 128, wgs, 12, 256) == kCost256x128Shares.f2 + kCost256x128Shares.s2 * 12);
  }
  // 200 workgroups of 16 steps: 56 idle units get through 46 bytes per ns for 4.1 us, not for the 8.3 of two tiles on a unit
  const AheadList l = list(12000000, 0, 0);
  CHECK(ahead_choice(&l, share_us(64, 64, 200, 16, 256), 64, 64, 56).workgroups == 0 && ahead_choice(&l, share_us(64, 64, 257, 16, 256), 64, 64, 56).workgroups == 56);
""")


def test_tiles_with_k_in_ranges_ask(tmp_path):
    """A launch whose tiles walk the ranges of K one after the other lasts that long and leaves most compute units idle: 333 x 704 x 3072, 66 tiles."""
    _run(tmp_path, r"""
  CHECK(ranges_us(66, 3072, 256) == kPlainCosts[12].f1 + kPlainCosts[12].s1 * 48 && ranges_us(300, 3072, 256) == kPlainCosts[12].f2 + kPlainCosts[12].s2 * 48);
  const AheadList l = list(67000000, 33000000, 0);
  CHECK(ahead_choice(&l, ranges_us(66, 3072, 256), 333, 384, 190).workgroups == 190 && ahead_choice(&l, ranges_us(66, 3072, 256), 333, 384, 190).ranges.r[1].bytes == 0);
""")
