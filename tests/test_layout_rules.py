"""The rules that choose between two forms of a step (csrc/layout_select.hpp)
take the faster one at the sizes where both were timed (MI355X; us per step,
as the comments of the rules give them; differences under 1 % are left out)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# fields, bytes per element, MB of one population buffer: plane order, runs of 4
ORDER = [
    (1, 8, 122, 40.83, 45.08), (1, 8, 291, 105.22, 106.80), (1, 8, 635, 226.09, 229.17), (1, 8, 725, 263.24, 260.32),
    (1, 8, 801, 289.94, 285.54), (1, 8, 889, 323.77, 314.89), (1, 8, 1462, 536.63, 514.82),
    (1, 8, 2158, 791.23, 760.64), (1, 4, 276, 105.57, 107.62), (1, 4, 731, 279.40, 274.13),
    (1, 4, 1079, 414.97, 404.83), (1, 4, 1522, 585.29, 577.75), (1, 4, 2073, 828.17, 783.68),
    (1, 2, 1036, 548.56, 535.02), (2, 8, 852, 439.0, 453.0), (2, 8, 3233, 1801.54, 1769.08),
    (2, 8, 3858, 2160.10, 2113.84), (2, 4, 1075, 627.38, 635.91), (2, 4, 2158, 1298.15, 1272.02),
    (2, 2, 1288, 1032.99, 1050.91), (2, 2, 1784, 1420.92, 1441.10),
]


def rules(tmp_path, lines):
    """The values of C++ expressions over csrc/layout_select.hpp."""
    src, exe = tmp_path / "r.cpp", str(tmp_path / "r")
    src.write_text("#include <cstdio>\n#include \"layout_select.hpp\"\nint main() {\n  using namespace lbamd;\n"
                   + "".join('  std::printf("%%d\\n", int(%s));\n' % x for x in lines) + "}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "badchimp-cpp_amd", "csrc"), str(src), "-o",
                    exe], check=True, capture_output=True)
    return list(map(int, subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split()))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_block_order_is_the_faster_one(tmp_path):
    got = rules(tmp_path, ["plane_order(%d, %d, %d000000LL)" % r[:3] for r in ORDER])
    assert got == [int(r[3] < r[4]) for r in ORDER]


# fields, MB of both buffers, of what else a step reads or writes (the link table; density and velocity): plain,
# streaming stores
STORES = [
    (1, 14.9, 7.0, 6.82, 6.52), (1, 29.7, 7.0, 9.44, 10.85), (1, 24.1, 10.7, 6.69, 7.46), (1, 103.1, 24.4, 23.44, 26.34),
    (1, 176.5, 83.6, 40.97, 42.83), (1, 201.4, 44.8, 40.34, 41.32), (1, 121.4, 115.0, 41.41, 43.05),
    (1, 201.5, 89.6, 49.85, 47.95), (1, 246.9, 58.5, 56.37, 54.70), (1, 242.8, 115.0, 66.27, 61.26),
    (1, 353.0, 83.6, 81.88, 71.69), (1, 162.0, 153.4, 62.04, 55.27), (1, 32.1, 0, 6.74, 8.01),
    (1, 201.4, 0, 31.69, 36.53), (1, 403.0, 0, 73.69, 68.33), (1, 255.0, 0, 46.61, 49.48), (1, 265.0, 0, 53.53, 50.68),
    (2, 14.9, 0, 13.43, 11.96), (2, 32.1, 0, 13.22, 12.57), (2, 48.2, 0, 17.00, 16.39), (2, 29.6, 0, 17.09, 16.44),
    (2, 64.2, 0, 18.69, 19.42), (2, 118.3, 0, 31.52, 33.53), (2, 103.1, 0, 32.86, 34.15), (2, 82.4, 0, 36.62, 38.36),
    (2, 242.8, 0, 96.51, 101.15), (2, 493.9, 0, 139.86, 130.43),
    (2, 29.7, 7.0, 23.14, 22.90), (2, 59.2, 14.0, 33.57, 32.26), (2, 100.6, 22.4, 43.59, 42.10),
    (2, 164.8, 39.0, 86.78, 83.93), (2, 246.9, 58.5, 128.06, 122.50), (2, 705.9, 83.6, 248.03, 236.27),
]
# the same for calls of one step, which write density and velocity
STORES_1 = [
    (1, 243.0, 51.0, 63.59, 57.87), (1, 247.0, 26.0, 59.32, 53.95), (1, 255.0, 27.0, 61.58, 56.08),
    (1, 209.0, 88.0, 77.90, 73.71), (1, 203.0, 22.0, 40.52, 45.80), (1, 200.0, 42.0, 42.36, 48.56),
    (1, 165.0, 18.0, 33.50, 39.39),
]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_stores_are_the_faster_ones(tmp_path):
    got = rules(tmp_path, ["stream_stores(%d, %d, %d)" % (r[1] * 1e6, r[0], r[2] * 1e6) for r in STORES])
    assert got == [int(r[4] < r[3]) for r in STORES]
    got = rules(tmp_path, ["stream_stores(%d, %d, 0, %d)" % (r[1] * 1e6, r[0], r[2] * 1e6) for r in STORES_1])
    assert got == [int(r[4] < r[3]) for r in STORES_1]


# bytes per element, tiles, nodes: tiled, plain
TILES = [
    (8, 242, 18818, 1.88, 3.25), (8, 425, 29114, 2.80, 3.40), (8, 425, 59400, 3.20, 3.66),
    (8, 500, 35950, 2.97, 3.92), (8, 570, 78480, 3.62, 4.16), (8, 570, 62438, 3.80, 3.68),
    (8, 616, 66138, 3.79, 3.99), (8, 616, 49486, 3.70, 3.55), (8, 680, 72634, 3.59, 4.17),
    (8, 680, 44844, 3.62, 3.46), (8, 748, 101600, 3.69, 4.33), (8, 792, 109220, 4.56, 4.40),
    (8, 792, 65222, 4.29, 3.65), (8, 840, 94144, 4.51, 4.26), (8, 880, 72278, 4.39, 4.19),
    (8, 946, 130048, 4.44, 4.72), (8, 946, 77314, 4.43, 4.22), (8, 1034, 142240, 5.25, 5.12),
    (8, 1100, 91040, 5.18, 4.31), (8, 1620, 229120, 6.96, 6.60), (8, 2278, 190280, 8.60, 5.62),
    (4, 242, 18818, 1.45, 3.06), (4, 616, 41610, 2.62, 3.13), (4, 840, 58664, 2.96, 3.12),
    (4, 946, 130048, 2.94, 3.61), (4, 2278, 190280, 4.96, 4.33),
]


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_tiles_are_taken_where_they_are_faster(tmp_path):
    got = rules(tmp_path, ["tiles_pay(%d, %d, %d)" % r[:3] for r in TILES])
    assert got == [int(r[3] < r[4]) for r in TILES]


XCDS = r'''
#include "rowbuild.hpp"
#include <cstdio>
using namespace lbamd;
// box of x planes of ny x nz fluid cells: 1 where consecutive blocks share an XCD
// in long runs, 2 where every plane's blocks go to the XCDs in order, else 0
static int form(int nx, int ny, int nz) {
  std::vector<uint32_t> coord;
  for (int x = 0; x < nx; ++x)
    for (int y = 0; y < ny; ++y)
      for (int z = 0; z < nz; ++z) coord.push_back(uint32_t(x) << 22 | uint32_t(y) << 12 | uint32_t(z));
  const std::vector<uint8_t> xcd = block_xcd(coord);
  int64_t changes = 0, mids = 0;
  for (size_t b = 1; b < xcd.size(); ++b) changes += xcd[b] != xcd[b - 1];
  for (size_t b = 0; b < xcd.size(); ++b) {
    const int64_t mid = std::min<int64_t>(coord.size() - 1, 256 * b + 128), n = ny * nz;
    mids += xcd[b] == mid % n * 8 / n;
  }
  const int64_t nb = xcd.size(), run = std::min<int64_t>(32, (nb + 7) / 8);
  return changes == (nb - 1) / run ? 1 : mids == nb ? 2 : 0;
}
int main() {
  std::printf("%d %d %d %d %d %d %d\n", form(300, 1, 300), form(258, 1, 620), form(177, 1, 900), form(60, 30, 40),
              form(90, 37, 55), form(40, 32, 64), form(70, 60, 60));
}
'''


def test_blocks_of_thin_planes_go_to_the_xcds_in_long_runs(tmp_path):
    """Planes of 1.2, 2.4, 3.5, 4.7 and 7.9 blocks in runs of blocks, of 8 and 14 plane by plane."""
    src, exe = tmp_path / "x.hip", str(tmp_path / "x")
    src.write_text(XCDS)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "badchimp-cpp_amd", "csrc"), str(src), "-o", exe], check=True,
                   capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    assert out.split() == ["1", "1", "1", "1", "1", "2", "2"], out
