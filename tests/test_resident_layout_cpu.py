"""Indexing of the sweep with weights in registers (csrc/zr_resident_layout.h), checked on the host.  The hand-over copy: no 128-byte
line of it may hold elements of two row tiles or of two column tiles, for every batch up to 160 columns, every width a column
tile can have, one to three row tiles and a ragged last one.  The kernel reads the copy without cache invalidation, so a line
with two producers could be read before the second of them has stored.  An embedding column's last blocks: what they read twice
must count once in all."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zoph_rnn_amd", "csrc")
PROGRAM = r"""
#include <cmath>
#include <cstdio>
#include <vector>
#include "zr_resident_layout.h"
int main() {
  int bad = 0;
  const int widths[] = {16, 32, 64}, sizes[] = {8, 9, 20, 24};
  for (int H : sizes)
    for (int mb = 1; mb <= 160; ++mb)
      for (int width : widths) {
        const int columns = zr_resident_columns(mb);
        const long long slot = zr_resident_slot(H, mb);
        const int rows = (H + kResidentRows - 1) / kResidentRows * kResidentRows;
        if (columns < mb || (slot * 4) % 128) ++bad, std::printf("H %d mb %d: %d columns, slot %lld\n", H, mb, columns, slot);
        std::vector<int> owner((slot * 4 + 127) / 128, -1);
        bool shared = false;
        for (int k = 0; k < rows; ++k)
          for (int n = 0; n < mb; ++n) {
            const long long at = zr_resident_at(k, n, columns);
            if (at >= slot) { shared = true; continue; }
            int& o = owner[at * 4 / 128];
            const int me = k / kResidentRows * 1000 + n / width;
            if (o >= 0 && o != me) shared = true;
            o = me;
          }
        if (shared) ++bad, std::printf("H %d mb %d, tiles of %d columns: a line with two producers\n", H, mb, width);
      }
  // every weight of an embedding column counts once in all: size classes of the kernel, 16-column and wider form
  for (int H = 8; H <= 1024; ++H) {
    const int blocks = 4 * (H <= 128 ? 8 : H <= 256 ? 16 : H <= 512 ? 32 : 64);
    std::vector<double> total(H, 0.0);
    for (int block = 0; block < blocks; ++block)
      for (int e = 0; e < 4; ++e) {
        const int k = (4 * block < H - 4 ? 4 * block : H - 4) + e;
        const int halvings = zr_resident_embed_halvings(H, blocks, block, k);
        if (halvings < 0 || halvings > 60) ++bad, std::printf("H %d: %d halvings\n", H, halvings);
        total[k] += std::ldexp(1.0, -halvings);
      }
    for (int k = 0; k < H; ++k)
      if (std::fabs(total[k] - 1.0) > std::ldexp(1.0, -53)) ++bad, std::printf("H %d: weight %d counts %g times\n", H, k, total[k]);
  }
  return bad ? 1 : 0;
}
"""


def test_lines_have_one_producer_and_weights_count_once(tmp_path):
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-Wall", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
