// Several collide-stream steps of a small two-dimensional node list in one launch.
//
// A step of a small list is bound by latency, not by bytes: the launch, the
// chain from a cell to its window words to its gathers, the stores.  Here a
// workgroup advances a tile of the box kTileSteps steps: it holds the tile with a
// halo of kTileSteps - 1 cells, one thread per cell, gathers the first step's
// populations from memory like the plain step, hands the post-collision values
// of the steps between through LDS, and stores the last step's of the tile's own
// cells.  The halo's cells are computed by every tile that needs them, each step
// one layer less.  The arithmetic and its operands are the plain step's, so the
// values are the same bits.
// 22 x 22 threads for 6 steps (tiles of 12 x 12 cells, 70 KB of LDS in FP64, two
// workgroups per CU) measured best of 2 to 8 steps and edges of 16 to 30.  us per
// step, tiled / plain: FP64 channel 64x48 1.54 / 2.95, 256x128 (32 k nodes) 2.1 /
// 3.3, 384x190 2.95 / 4.0, 512x256 (946 tiles) 4.4 / 4.6; FP32S 256x128 1.6 / 2.9,
// 512x256 2.9 / 3.5.  Larger boxes, and those with many solids, pay more for the
// halos' work than a launch costs (tiles_pay in layout_select.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include "addressing.hpp"
#include "lattice.hpp"

namespace lbamd {

constexpr int kTileSteps = 6;
constexpr int kTileEdge = 22;                           // threads along each axis
constexpr int kTileCells = kTileEdge - 2 * (kTileSteps - 1);  // own cells along each axis

// The box of a tiled launch: cells along x and along the rows, and whether x is
// periodic.
struct TileBox {
  int32_t EX, EZ, periodic;
  __host__ __device__ int32_t tiles_z() const { return (EZ + kTileCells - 1) / kTileCells; }
  __host__ __device__ int32_t tiles() const { return (EX + kTileCells - 1) / kTileCells * tiles_z(); }
};

// collide(f, i): the post-collision values of node i in place of its
// pre-collision ones.
template <typename T, class Collide>
__device__ __forceinline__ void tile_steps(const T* __restrict__ fin, T* __restrict__ fout, const RowWin& ad,
                                           const TileBox& box, Collide&& collide) {
  using L = D2Q9;
  constexpr int Q = L::nQ, H = kTileSteps - 1, E = kTileEdge;
  __shared__ T post[2][Q][E * E];
  const int32_t t = static_cast<int32_t>(threadIdx.x), lx = t / E, lz = t % E;
  const int32_t nz = box.tiles_z(), tile = static_cast<int32_t>(blockIdx.x);
  const int32_t x = tile / nz * kTileCells + lx - H, Z = tile % nz * kTileCells + lz - H;
  // layers of the tile's box around this cell
  const int32_t depth = min(min(lx, E - 1 - lx), min(lz, E - 1 - lz));
  int32_t X = x;
  if (box.periodic) {
    X = x % box.EX;
    if (X < 0) X += box.EX;
  }
  bool active = X >= 0 && X < box.EX && Z >= 0 && Z < box.EZ;
  uint32_t from = 0u;  // bit q: the source of direction q is fluid
  int32_t i = 0;
  T f[Q];
  if (active) {
    RowWin::Rows<L> r;
    ad.template cell_rows<L>((static_cast<uint32_t>(X) << 22) | static_cast<uint32_t>(Z), r);
    active = (r.m[1] >> (r.t + 1u)) & 1u;
    if (active) {
      i = static_cast<int32_t>(r.b0[1]);
      uint32_t src[Q - 1];
      RowWin::row_sources<L>(i, r, src);
#pragma unroll
      for (int q = 0; q < Q - 1; ++q) {
        f[q] = ld_elem<true>(fin, src[q]);
        from |= r.fluid(q) & (1u << q);
      }
      f[Q - 1] = ld_elem<true>(fin, pidx<Q>(Q - 1, i));
    }
  }
#pragma unroll
  for (int s = 0; s < kTileSteps; ++s) {
    const bool now = active && depth >= s;
    if (now) collide(f, i);
    if (s == kTileSteps - 1) {
      // own cells of the last tiles end with the box
      if (now && x < box.EX) {
        T* __restrict__ out = elem_ptr<true>(fout, pidx<Q>(0, i));
#pragma unroll
        for (int q = 0; q < Q; ++q) out[q << kPLog] = f[q];
      }
      break;
    }
    // (the step after the next writes this half again, behind the next barrier)
    T(&buf)[Q][E * E] = post[s & 1];
    if (now) {
#pragma unroll
      for (int q = 0; q < Q; ++q) buf[q][t] = f[q];
    }
    __syncthreads();
    if (active && depth > s) {
#pragma unroll
      for (int q = 0; q < Q - 1; ++q) {
        const int at = t - (L::c(q, 0) * E + L::c(q, 1));
        f[q] = (from >> q) & 1u ? buf[q][at] : buf[L::rev(q)][t];
      }
    }
  }
}

}  // namespace lbamd
