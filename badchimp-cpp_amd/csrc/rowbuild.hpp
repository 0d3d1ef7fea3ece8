// Host-side construction of the row layouts (addressing.hpp: RowAddr, RowWin).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <string>
#include <utility>
#include <vector>

#include "../../include/badchimp_amd.h"
#include "addressing.hpp"
#include "host_threads.hpp"
#include "lattice.hpp"

namespace lbamd {

// Rows are ordered in tiles of 2^kTileLogX x 2^kTileLogY (X, Y) columns.
// Runs of 32 rows along Y measured best on the 256^3 pack (33.0 GLUPS FP32S,
// against 31.6 for 8 x 8 tiles with blocks remapped per XCD and 32.9 with no
// tiles); the differences between tile shapes are small.
constexpr int kTileLogX = 0;
constexpr int kTileLogY = 5;

// Cartesian row layout of the bulk nodes (see addressing.hpp): the box, the
// compact order (tiled row order), the packed cell of each compact node and
// {base, mask} per (row, 32-cell word).
struct RowBuild {
  RowGeom g{};
  int32_t lo[3] = {0, 0, 0};    // rows_from_geometry: geometry cell of box coordinate 0
  std::vector<int32_t> order;   // compact index -> bulk index
  std::vector<uint32_t> coord;  // compact index -> packed cell
  std::vector<uint2> rows;
};

// The row layout straight from a geometry (C order over x, y[, z]; cells > 0
// are fluid), without a neighbour index: the fluid cells in tiled row order,
// which is the order build_rows gives the node list that the vtklb writer
// makes of the same geometry.  Periodic axes span the whole box; closed axes
// span the fluid cells' extent.
inline bool rows_from_geometry(int lattice, const int32_t* dims, const int32_t* geo, int32_t periodic_mask,
                               RowBuild& rb, std::string& why) {
  const int nD = lattice == LB_D2Q9 ? 2 : 3;
  // geometry axis of row axis a (X, Y, Z), -1 for the missing Y of 2-D
  const int ax[3] = {0, nD == 3 ? 1 : -1, nD == 3 ? 2 : 1};
  int64_t ncell = 1;
  for (int d = 0; d < nD; ++d) {
    if (dims[d] < 1) { why = "empty geometry"; return false; }
    ncell *= dims[d];
  }
  int32_t D[3], lo[3], hi[3];
  for (int a = 0; a < 3; ++a) {
    D[a] = ax[a] < 0 ? 1 : dims[ax[a]];
    lo[a] = D[a];
    hi[a] = -1;
  }
  const int64_t sy = nD == 3 ? dims[2] : 1, sx = nD == 3 ? static_cast<int64_t>(dims[1]) * dims[2] : dims[1];
  auto at = [&](int32_t X, int32_t Y, int32_t Z) -> int64_t {  // geometry index of row-axis cell
    return nD == 3 ? X * sx + Y * sy + Z : X * sx + Z;
  };
  int64_t nfluid = 0;
  for (int32_t x = 0; x < D[0]; ++x)
    for (int32_t y = 0; y < D[1]; ++y)
      for (int32_t z = 0; z < D[2]; ++z)
        if (geo[at(x, y, z)] > 0) {
          ++nfluid;
          const int32_t p[3] = {x, y, z};
          for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], p[a]);
            hi[a] = std::max(hi[a], p[a]);
          }
        }
  if (nfluid == 0) { why = "no fluid cells"; return false; }
  for (int a = 0; a < 3; ++a) rb.lo[a] = lo[a];
  RowGeom& g = rb.g;
  g.periodic = 0;
  for (int a = 0; a < 3; ++a) {
    const bool per = ax[a] >= 0 && ((periodic_mask >> ax[a]) & 1);
    g.E[a] = per ? D[a] : hi[a] - lo[a] + 1;
    if (per) g.periodic |= 1 << a;
  }
  if (g.E[0] > 1024 || g.E[1] > 1024 || g.E[2] > 4096) { why = "box too large for packed coordinates"; return false; }
  g.lx = kTileLogX;
  g.ly = g.E[1] >= (1 << kTileLogY) ? kTileLogY : 0;
  const int32_t nTx = (g.E[0] + (1 << g.lx) - 1) >> g.lx;
  g.nTy = (g.E[1] + (1 << g.ly) - 1) >> g.ly;
  g.W = (g.E[2] + 31) / 32;
  const int64_t R = static_cast<int64_t>(nTx) * g.nTy << (g.lx + g.ly);
  rb.order.clear();
  rb.coord.clear();
  rb.coord.reserve(static_cast<size_t>(nfluid));
  rb.rows.assign(static_cast<size_t>(R) * g.W, uint2{0u, 0u});
  // cell of the box coordinate v along row axis a
  auto cellc = [&](int a, int32_t v) { return (g.periodic >> a) & 1 ? (v + lo[a]) % D[a] : v + lo[a]; };
  for (int32_t tx = 0; tx < nTx; ++tx)
    for (int32_t ty = 0; ty < g.nTy; ++ty)
      for (int32_t ix = 0; ix < (1 << g.lx); ++ix)
        for (int32_t iy = 0; iy < (1 << g.ly); ++iy) {
          const int32_t X = (tx << g.lx) | ix, Y = (ty << g.ly) | iy;
          if (X >= g.E[0] || Y >= g.E[1]) continue;
          const size_t r = static_cast<size_t>(g.row(X, Y));
          const int32_t cx0 = cellc(0, X), cy0 = cellc(1, Y);
          for (int32_t Z = 0; Z < g.E[2]; ++Z) {
            if (geo[at(cx0, cy0, cellc(2, Z))] <= 0) continue;
            rb.coord.push_back((static_cast<uint32_t>(X) << 22) | (static_cast<uint32_t>(Y) << 12) |
                               static_cast<uint32_t>(Z));
            rb.rows[r * g.W + (Z >> 5)].y |= 1u << (Z & 31);
          }
        }
  uint32_t run = 0;
  for (auto& e : rb.rows) {
    e.x = run;
    run += static_cast<uint32_t>(__builtin_popcount(e.y));
  }
  return true;
}

// Row windows (addressing.hpp, RowWin and RowWinZ): for the halo-padded row
// (X+1, Y+1) and word w, the compact index of the first fluid cell at or after
// 8w (from node 0, or from the first node of the x plane) and the fluid bits
// of cells 8w-1 .. 8w+8.  Halo rows of a periodic axis repeat the rows they
// wrap to; those of a closed axis stay empty.
struct WinBuild {
  std::vector<uint32_t> win;
  std::vector<uint32_t> plane;  // first node of each padded X; empty: bases from node 0
  std::vector<uint32_t> count;  // fluid cells of each padded row (box periodic along the row axis)
  int32_t PY = 0, W = 0, EZ = 0;
};

// planes: bases from the first node of the x plane also where the node list
// fits without (for tests).  threads: large tables are filled on host threads;
// false for a caller that is one of several threads with a geometry each.
inline bool build_windows(const RowBuild& rb, bool allow_periodic, WinBuild& wb, std::string& why,
                          bool planes = false, bool threads = true) {
  const RowGeom& g = rb.g;
  const bool pz = (g.periodic & 4) != 0;
  if (pz && !allow_periodic) {
    why = "periodic along the row axis";
    return false;
  }
  constexpr uint32_t kMax = 1u << kWinBase;
  const int32_t PX = g.E[0] + 2, EZ = g.E[2];
  wb.PY = g.E[1] + 2;
  wb.W = win_words(EZ);
  wb.EZ = EZ;
  wb.win.assign(static_cast<size_t>(PX) * wb.PY * wb.W, 0u);
  wb.count.assign(pz ? static_cast<size_t>(PX) * wb.PY : 0u, 0u);
  wb.plane.assign(planes || rb.coord.size() >= kMax ? static_cast<size_t>(PX) : 0u, 0u);
  // the nodes of a plane are consecutive (one plane per tile along X)
  static_assert(kTileLogX == 0, "x planes are not consecutive in the compact order");
  std::atomic<bool> fits{true};
  auto plane = [&](int32_t px) {
    int32_t X = px - 1;
    if (!RowGeom::wrap(X, g.E[0], g.periodic & 1)) return;
    const uint32_t base = wb.plane.empty() ? 0u : rb.rows[static_cast<size_t>(g.row(X, 0)) * g.W].x;
    if (!wb.plane.empty()) wb.plane[px] = base;
    for (int32_t py = 0; py < wb.PY; ++py) {
      int32_t Y = py - 1;
      if (!RowGeom::wrap(Y, g.E[1], g.periodic & 2)) continue;
      const uint2* words = &rb.rows[static_cast<size_t>(g.row(X, Y)) * g.W];  // 32 cells each, no bits beyond E_Z
      const size_t pr = static_cast<size_t>(px) * wb.PY + py;
      uint32_t* out = &wb.win[pr * wb.W];
      const uint32_t row0 = words[0].y & 1u, rowN = (words[g.W - 1].y >> ((EZ - 1) & 31)) & 1u;
      uint32_t before = pz ? rowN : 0u;  // the cell before the word
      for (int32_t k = 0; k < g.W; ++k) {
        const uint32_t y = words[k].y, next = k + 1 < g.W ? words[k + 1].y & 1u : 0u;
        uint32_t first = words[k].x - base;
        for (int32_t w = 4 * k; w < std::min(4 * k + 4, wb.W); ++w) {
          const int32_t h = (w & 3) << kWinLog;
          const uint32_t cells = (y >> h) & 0xffu;
          const uint32_t after = h < 24 ? (y >> (h + 8)) & 1u : next;
          uint32_t bits = before | (cells << 1) | (after << 9);
          // the cell after the row's last one is its first
          if (pz && w == wb.W - 1) bits |= row0 << (EZ - (w << kWinLog) + 1);
          if (first >= kMax) fits = false;
          out[w] = (bits << kWinBase) | (first & (kMax - 1u));
          first += static_cast<uint32_t>(__builtin_popcount(cells));
          before = cells >> 7;
        }
      }
      if (pz) wb.count[pr] = words[g.W - 1].x + static_cast<uint32_t>(__builtin_popcount(words[g.W - 1].y)) - words[0].x;
    }
  };
  // (parallel_ranges counts items of about a cell's work)
  const int64_t per = static_cast<int64_t>(wb.PY) * wb.W;
  auto fill = [&](int64_t b, int64_t e, int) {
    for (int64_t px = (b + per - 1) / per; px * per < e; ++px) plane(static_cast<int32_t>(px));
  };
  if (threads) parallel_ranges(PX * per, fill);
  else fill(0, PX * per, 0);
  if (!fits) {
    why = "x plane above 2^22 nodes";
    return false;
  }
  return true;
}

// The cells around compact node i as RowWin and RowWinZ find them on the device.
struct WinNode {
  const WinBuild& wb;
  const int64_t i;
  const int32_t X, Z;
  const size_t pr;    // padded row
  const uint32_t t;   // bit of cell z - 1 in a word
  WinNode(const RowBuild& rb, const WinBuild& w, int64_t n)
      : wb(w), i(n), X(static_cast<int32_t>(rb.coord[n] >> 22)), Z(static_cast<int32_t>(rb.coord[n] & 4095u)),
        pr(static_cast<size_t>(X + 1) * w.PY + (((rb.coord[n] >> 12) & 1023u) + 1)),
        t(kWinBase + (static_cast<uint32_t>(Z) & (kWinCells - 1u))) {}
  // the cell (dx, dy, dz) off the node's: {fluid, compact index}, or {false, i}
  std::pair<bool, int64_t> cell(int dx, int dy, int dz) const {
    const size_t row = pr + static_cast<int64_t>(dx) * wb.PY + dy;
    const uint32_t m = wb.win[row * wb.W + (Z >> kWinLog)];
    if (!((m >> (t + 1 + dz)) & 1u)) return {false, i};
    const uint32_t below = (2u << t) - (2u << kWinBase);
    const uint32_t b0 = (m & ((1u << kWinBase) - 1u)) + static_cast<uint32_t>(__builtin_popcount(m & below)) +
                        (wb.plane.empty() ? 0u : wb.plane[X + 1 + dx]);
    if (dz == 0) return {true, static_cast<int64_t>(b0)};
    const uint32_t n = !wb.count.empty() && Z == (dz < 0 ? 0 : wb.EZ - 1) ? wb.count[row] : 0u;
    if (dz < 0) return {true, static_cast<int64_t>(b0 - 1u + n)};
    return {true, static_cast<int64_t>(b0 + ((m >> (t + 1u)) & 1u) - n)};
  }
};

// Source of direction q for compact node i under the row windows.
inline std::pair<bool, int64_t> win_source(int lattice, const RowBuild& rb, const WinBuild& wb, int q, int32_t i) {
  const WinNode n(rb, wb, i);
  if (lattice == LB_D2Q9) return n.cell(-D2Q9::c(q, 0), 0, -D2Q9::c(q, 1));
  return n.cell(-D3Q19::c(q, 0), -D3Q19::c(q, 1), -D3Q19::c(q, 2));
}

// XCD of each 256-node block of a node list in row order, for dispatch (the
// hardware hands workgroup k to XCD k mod 8, and each XCD has its own L2).  A
// block's gathers reach the planes x-1, x and x+1 near its own rows.  So each
// plane is cut into 8 runs of about equal length along its rows, and run k of
// every plane goes to XCD k: the rows that a gather reaches, and the node's own
// lines that its bounce-back reads, were read or will be by the same XCD.  On
// the 256^3 pack in FP32S the L2s then fetch 1.11x the populations instead of
// 1.55x (node_block: runs of 4 blocks round-robin).  Planes of fewer than 8 blocks
// on average have runs shorter than a block, so that a block reaches into several
// of them: there an XCD takes runs of consecutive blocks, long ones (n / 8 blocks,
// at most 32), which hold several planes.  Runs of 32 / plane by plane / runs of 4,
// us per step by blocks per plane: D2Q9 channel FP64 258x620 (2.4) 5.36 / 8.18 /
// 6.51, 177x900 (3.5) 5.42 / 8.14 / 7.44, 106x1500 (5.9) 5.51 / 5.91 / 8.02; FP32S
// 258x620 4.06 / 4.91 / 4.60, 1000x1900 (7.4) 23.2 / 24.8 / 24.4; packs FP64
// 90x28x28 open (2.6) 4.92 / 6.48 / 5.29, 48^3 (3.6) 5.00 / 5.18 / 5.32, 64^3 (6)
// 7.2 / 7.9 / 8.8, 74^3 (8) 11.20 / 11.25 / 11.86; FP32S 900x56x56 (4.6) 27.1 / 31.6
// / 32.9; from 8 on 80^3 (9.3) FP32S 7.71 / 7.70, FP16S 6.57 / 6.49, 32x64x64 open
// (15) FP64 8.4 / 7.9.  In a batch, where the items of all solves share the XCDs,
// the plane order pays from two blocks per plane on (24 solves of 32^3 to 128^3, 300
// steps: 68.1 ms for 69.0).
constexpr int64_t kPlaneBlocks = 8, kBatchPlaneBlocks = 2;
inline std::vector<uint8_t> block_xcd(const std::vector<uint32_t>& coord, int64_t plane_blocks = kPlaneBlocks) {
  const int64_t n = static_cast<int64_t>(coord.size()), nb = (n + kBlock - 1) / kBlock;
  std::vector<uint8_t> xcd(static_cast<size_t>(nb));
  std::vector<int64_t> start;  // first node of each plane
  for (auto it = coord.begin(); it != coord.end(); it = std::upper_bound(it, coord.end(), *it | 0x3fffffu))
    start.push_back(it - coord.begin());
  if (nb < plane_blocks * static_cast<int64_t>(start.size())) {
    const int64_t run = std::min<int64_t>(32, (nb + 7) / 8);
    for (int64_t b = 0; b < nb; ++b) xcd[b] = static_cast<uint8_t>((b / run) % 8);
    return xcd;
  }
  start.push_back(n);
  size_t p = 0;
  for (int64_t b = 0; b < nb; ++b) {
    const int64_t mid = std::min(n - 1, b * kBlock + kBlock / 2);
    while (start[p + 1] <= mid) ++p;
    xcd[b] = static_cast<uint8_t>((mid - start[p]) * 8 / (start[p + 1] - start[p]));
  }
  return xcd;
}

// Items in an order that hands each to its XCD: position k is taken by the
// next item of XCD k mod 8; what an XCD has beyond its positions goes, in
// order, where others have fewer.
template <typename T>
std::vector<T> interleave_xcds(const std::vector<T>& items, const std::vector<uint8_t>& xcd) {
  const size_t n = items.size();
  std::vector<T> out(n), rest;
  size_t at[8];
  for (size_t x = 0; x < 8; ++x) at[x] = x;
  for (size_t k = 0; k < n; ++k) {
    size_t& p = at[xcd[k]];
    if (p < n) out[p] = items[k];
    else rest.push_back(items[k]);
    p += 8;
  }
  size_t r = 0;
  for (size_t x = 0; x < 8; ++x)
    for (size_t p = at[x]; p < n; p += 8) out[p] = rest[r++];
  return out;
}

// Block order of a node list in row order (RowWin::order).  Empty for lists
// of fewer than 64 blocks.
inline std::vector<int32_t> block_order(const std::vector<uint32_t>& coord) {
  const std::vector<uint8_t> xcd = block_xcd(coord);
  if (xcd.size() < 64) return {};
  std::vector<int32_t> blocks(xcd.size());
  for (size_t b = 0; b < blocks.size(); ++b) blocks[b] = static_cast<int32_t>(b);
  return interleave_xcds(blocks, xcd);
}

}  // namespace lbamd
