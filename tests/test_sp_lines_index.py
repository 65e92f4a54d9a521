"""The points of SP's staged line tasks (csrc/sp_lines_index.h) against the
plain definition, on the CPU: lines numbered across then up, in zones whose
cross extent is smaller than a task, a few points, or millions (the index of
a line wraps by comparison, exact for any extent)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include <initializer_list>
#define __host__
#define __device__
#define __forceinline__ inline
#include "sp_lines_index.h"
using namespace npbmz::sp;

template <int DIR>
int check(int nx, int ny, int nz) {
  const int across = (DIR == 0 ? ny : nx) - 2, up = (DIR == 2 ? ny : nz) - 2;
  const int nl = DIR == 0 ? nx : DIR == 1 ? ny : nz;
  const int lines = across * up;
  int bad = 0;
  for (int first = 0; first < lines; first += kStageLines) {
    // of large extents, the tasks around each wrap and some in between
    const int a = first % across;
    if (across > 5000 && a > 20 && a < across - 20 && first / kStageLines % 50021) continue;
    const StagedLines<DIR> G(nx, ny, nz, first);
    const int cnt = lines - first < kStageLines ? lines - first : kStageLines;
    if (G.cnt != cnt || G.nl != nl) return 1;
    for (int e = 0; e < cnt * nl; ++e) {
      const int eli = DIR == 0 ? e / nl : e % cnt, eq = DIR == 0 ? e % nl : e / cnt;
      const int line = first + eli, x = 1 + line % across, y = 1 + line / across;
      const int i = DIR == 0 ? eq : x, j = DIR == 0 ? x : DIR == 1 ? eq : y, k = DIR == 2 ? eq : y;
      int li, q;
      const int p = G.at(e, li, q);
      bad += li != eli || q != eq || p != (k * ny + j) * nx + i;
    }
  }
  return bad;
}

int main() {
  const int n[] = {5, 6, 7, 8, 9, 13, 38, 104, 310};
  int bad = 0;
  for (int nx : n) for (int ny : n) for (int nz : n) {
    if (nx * ny * nz > 400000) continue;
    if (nx >= 6) bad += check<0>(nx, ny, nz);
    if (ny >= 6) bad += check<1>(nx, ny, nz);
    if (nz >= 6) bad += check<2>(nx, ny, nz);
  }
  // the cross extent in the millions, up to the largest zone (2^30 points)
  for (int wide : {1048573, 1048579, 6556022, 6556025, 16777219, 29826161}) {
    bad += check<0>(6, wide, 6);
    bad += check<1>(wide, 6, 6);
    bad += check<2>(wide, 6, 6);
  }
  std::printf("%d\n", bad);
  return bad != 0;
}
"""


def test_staged_lines_index_every_point_once_and_in_order(tmp_path):
    src = tmp_path / "check.cpp"
    src.write_text(SOURCE)
    exe = tmp_path / "check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I",
                    os.path.join(ROOT, "npbapps.jl_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
