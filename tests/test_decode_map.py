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
int main(int argc, char** argv) {
  for (int i = 1; i + 3 < argc; i += 4) {
    const int dh = atoi(argv[i]), B = atoi(argv[i + 1]), H = atoi(argv[i + 2]), nsplit = atoi(argv[i + 3]), blocks = B * H * nsplit;
    std::vector<int> seen((size_t)blocks);
    for (int id = 0; id < blocks; ++id) {
      const DecodeSlot t = decode_by_length(dh, B, H) ? decode_slot_by_length(id, B, H, nsplit) : decode_slot_by_pair(id, B, H, nsplit);
      if (t.s < 0 || t.s >= nsplit || t.h < 0 || t.h >= H || t.seq < 0 || t.seq >= B) { printf("%d %d %d %d: workgroup %d outside\n", dh, B, H, nsplit, id); return 1; }
      if (seen[((size_t)t.seq * H + t.h) * nsplit + t.s]++) { printf("%d %d %d %d: workgroup %d takes a part twice\n", dh, B, H, nsplit, id); return 1; }
    }
    for (int group : {1, 2, 4})
      for (int n = 0; n < 5000; n += 1 + n / 50) {
        const int r = decode_ranges(dh, group, B, H, nsplit, n);
        if (r < 1 || r > nsplit || (r > 1 && (r - 1) * 128 >= n)) { printf("%d %d %d %d: %d keys in %d ranges\n", dh, B, H, nsplit, n, r); return 1; }
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
                           f"static_assert(t{len(asserts)}.s == {s} && t{len(asserts)}.h == {pair % H} && t{len(asserts)}.seq == {pair // H});")
    _build(tmp_path, '#include "decode_map.hpp"\nusing namespace fsvd;\n' + "\n".join(asserts) + "\nint main() { return 0; }\n")
