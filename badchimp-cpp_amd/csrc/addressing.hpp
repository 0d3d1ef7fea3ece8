// Where a bulk node pulls each population from: the address layouts.
//
// Every layout provides sources<L>(i, src): the population element index
// (pidx, context.hpp) of the post-collision value that becomes f_q of node i,
// for q = 0..Q-2 (the rest direction always reads itself).  A stream link
// gives (q, j) with j the compact index of the upwind neighbour; a link from
// a solid gives (rev q, i), the half-way bounce-back.  Each layout first
// issues all its addressing loads and then does the arithmetic, so that the
// loads are in flight together.
//
// TableAddr  one 32-bit link per (direction, node): kind + index (see
//            context.hpp).  Works for any node list, including fluid links to
//            the ghost node 0.  4 B per link per step.
//
// RowAddr    the bulk nodes are cells of a Cartesian box, cut into rows along
//            the last axis (z in 3-D, y in 2-D).  Per row and 32-cell word it
//            keeps {base, mask}: the fluid bit mask and the compact index of
//            the word's first fluid cell.  A node stores only its packed cell
//            coordinate (4 B); the source cell r - c_q (periodic axes wrap) is
//            fluid if its bit is set, and then its compact index is base +
//            popcount(mask below the bit).  The table is a few MB and stays in
//            L2 / MALL.  One lookup per direction.
//
// RowWin     per row and word w of 8 cells it keeps, in one 32-bit word, the
//            fluid bits of the 10 cells 8w-1 .. 8w+8 (bit kWinBase+k: cell
//            8w-1+k) and the compact index of the first fluid cell at or after
//            8w.  The node's own word then covers the cells z-1, z, z+1 of
//            every neighbouring row, so the 9 (D3Q19) or 3 (D2Q9) neighbouring
//            rows are one 4-byte load each, and the three sources in a row
//            follow from one popcount: with b0 the index of the first fluid
//            cell at or after z, the source at z is b0, at z-1 it is b0-1, at
//            z+1 it is b0 + bit(z).  The window table has a halo of rows, so
//            no wrap logic runs per node.  22 bits hold the index of up to
//            4.19 M nodes; larger node lists count it from the first node of
//            the cell's x plane, three more loads per node.
//            One dword per row and not more: a wave's load of up to 4 bytes
//            per lane takes the vector L1 about 5 cycles where 16 lanes read
//            neighbouring words (the nodes of a row do), one of 8 or 16 bytes
//            takes 17 whatever it reads (measured on tables in L2), and the
//            step keeps that unit busy 79-87 % of its time.  Against 16-byte
//            entries over 32 cells a step takes, on the 256^3 pack, 127 us for
//            142 (FP16S), 187 for 192 (FP32S) and 350 as before (FP64, bound
//            by the memory); on a 161 x 143 x 150 pack 26.8 for 30.1 (FP16S).
//            The struct is kept small: 16 bytes more made the step of the
//            256 x 128 channel 4 % slower, which waits for its arguments.
// RowWinZ    RowWin for boxes that are periodic along the row axis: the bits of
//            the first and the last word wrap, and the nodes at z = 0 and
//            z = E_Z - 1 read the neighbouring rows' fluid counts, by which
//            the compact index steps at the wrap.
//
// Rows are ordered in tiles of 2^lx x 2^ly rows, which keeps the neighbour
// rows of a tile close in the compact order.  The row layouts are validated on
// the host against the neighbour index and switched on only when every link
// they compute equals the table's.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "context.hpp"

namespace lbamd {

// Block order: the hardware hands consecutive workgroups to the eight XCDs
// round-robin.  node_block() gives each XCD runs of kXcdChunk consecutive
// 256-node blocks, so neighbouring rows are mostly read through one L2, while
// all CUs still sweep one compact front whose halo stays in the shared MALL.
// On the 256^3 pack runs of 4 blocks are 2.4 % faster than runs of 1 (the
// plain order) in FP32S and 2 % in FP64; runs of 8-32 give about the same,
// one contiguous range per XCD (eight fronts) is 3 % slower.  It serves the
// link table, the rows and the largest lists (plane_order in layout_select.hpp);
// the other row windows and the batched items go to the XCDs plane by plane
// (block_order, interleave_xcds in rowbuild.hpp).  The mapping only changes which
// workgroup computes a block: per-block partial sums keep their block index, so
// results do not change.
constexpr int32_t kXcdChunk = 4;
__device__ __forceinline__ int32_t node_block(int32_t b, int32_t nb) {
  const int32_t full = (nb / (8 * kXcdChunk)) * (8 * kXcdChunk);
  if (b >= full) return b;  // the tail keeps the plain order
  const int32_t xcd = b & 7, k = b >> 3;
  return ((k / kXcdChunk) * 8 + xcd) * kXcdChunk + (k % kXcdChunk);
}

// Block of workgroup wg of nb: the layout's block order where it has one
// (block_order in rowbuild.hpp), else node_block.
template <class A>
__device__ __forceinline__ int32_t block_of(const A& ad, int32_t wg, int32_t nb) {
  if constexpr (A::kOrdered) {
    if (ad.order) return ad.order[wg];
  }
  return node_block(wg, nb);
}
// The same with the dispatch order reversed: a pass that follows another one over
// the same nodes starts where the first one ended, so its first reads find the
// lines that the first pass fetched last still in the MALL.  The two-phase
// collision pass runs this way after the colour pass.
template <class A>
__device__ __forceinline__ int32_t block_of_rev(const A& ad, int32_t wg, int32_t nb) {
  return block_of(ad, nb - 1 - wg, nb);
}

// Element indices are 32-bit: a context keeps Q * NP * fields below 2^32.
// kOff32: the layout is only used for population buffers below 4 GiB, so the
// kernels may address them with 32-bit byte offsets from the buffer base.
struct TableAddr {
  static constexpr bool kOff32 = false, kOrdered = false;
  const uint32_t* __restrict__ link;
  uint32_t NP;
  template <class L>
  __device__ __forceinline__ void sources(int32_t i, uint32_t (&src)[L::nQ - 1]) const {
    uint32_t l[L::nQ - 1];
#pragma unroll
    for (int q = 0; q < L::nQ - 1; ++q) l[q] = link[static_cast<uint64_t>(q) * NP + i];
#pragma unroll
    for (int q = 0; q < L::nQ - 1; ++q) {
      const uint32_t kind = l[q] >> 30;
      const uint32_t j = l[q] & kLinkIndexMask;
      // stream: (q, j); bounce: (rev q, i); ghost 0: (rev q, j) -- one index
      // computation on selected operands, no branch
      const uint32_t jj = kind == kLinkBounce ? static_cast<uint32_t>(i) : j;
      const uint32_t qq = kind == kLinkStream ? static_cast<uint32_t>(q) : static_cast<uint32_t>(L::rev(q));
      src[q] = pidx<L::nQ>(qq, jj);
    }
  }
};

struct RowGeom {
  int32_t E[3];      // box extent along X, Y, Z (2-D: X = x, Y = 1, Z = y)
  int32_t periodic;  // bit 0 X, bit 1 Y, bit 2 Z
  int32_t lx, ly;    // tile of 2^lx x 2^ly rows
  int32_t nTy, W;    // tiles along Y, 32-bit words per row
  // row index of cell column (X, Y)
  __host__ __device__ __forceinline__ int32_t row(int32_t X, int32_t Y) const {
    return (((X >> lx) * nTy + (Y >> ly)) << (lx + ly)) | ((X & ((1 << lx) - 1)) << ly) |
           (Y & ((1 << ly) - 1));
  }
  // wrap one coordinate into [0, E); false when it leaves a non-periodic box
  __host__ __device__ static __forceinline__ bool wrap(int32_t& v, int32_t E, bool periodic) {
    if (v >= 0 && v < E) return true;
    v += v < 0 ? E : -E;
    return periodic;
  }
};

// Cells of a row window's word, and the bits of its base.
constexpr uint32_t kWinLog = 3;
constexpr uint32_t kWinCells = 1u << kWinLog;
constexpr uint32_t kWinBase = 22;
__host__ __device__ __forceinline__ constexpr int32_t win_words(int32_t ez) {
  return (ez + static_cast<int32_t>(kWinCells) - 1) >> kWinLog;
}

// lattice direction components mapped to (X, Y, Z)
template <class L>
__host__ __device__ __forceinline__ constexpr int cx(int q) { return L::c(q, 0); }
template <class L>
__host__ __device__ __forceinline__ constexpr int cy(int q) { return L::nD == 3 ? L::c(q, 1) : 0; }
template <class L>
__host__ __device__ __forceinline__ constexpr int cz(int q) { return L::nD == 3 ? L::c(q, 2) : L::c(q, 1); }

struct RowAddr {
  static constexpr bool kOff32 = false, kOrdered = false;
  const uint32_t* __restrict__ coord;  // X << 22 | Y << 12 | Z
  const uint2* __restrict__ rows;      // {base, mask} per (row, word)
  uint32_t NP;
  RowGeom g;
  template <class L>
  __device__ __forceinline__ void sources(int32_t i, uint32_t (&src)[L::nQ - 1]) const {
    const uint32_t c = coord[i];
    const int32_t X0 = static_cast<int32_t>(c >> 22), Y0 = static_cast<int32_t>((c >> 12) & 1023u),
                  Z0 = static_cast<int32_t>(c & 4095u);
    uint2 e[L::nQ - 1];
    uint32_t bit[L::nQ - 1];
#pragma unroll
    for (int q = 0; q < L::nQ - 1; ++q) {
      int32_t X = X0 - cx<L>(q), Y = Y0 - cy<L>(q), Z = Z0 - cz<L>(q);
      bool inside = true;
      if (cx<L>(q) != 0) inside = RowGeom::wrap(X, g.E[0], g.periodic & 1) && inside;
      if (cy<L>(q) != 0) inside = RowGeom::wrap(Y, g.E[1], g.periodic & 2) && inside;
      if (cz<L>(q) != 0) inside = RowGeom::wrap(Z, g.E[2], g.periodic & 4) && inside;
      const int64_t slot = inside ? static_cast<int64_t>(g.row(X, Y)) * g.W + (Z >> 5) : 0;
      e[q] = rows[slot];
      bit[q] = inside ? (1u << (Z & 31)) : 0u;
    }
#pragma unroll
    for (int q = 0; q < L::nQ - 1; ++q) {
      const uint32_t m = 0u - static_cast<uint32_t>((e[q].y & bit[q]) != 0u);
      const uint32_t j = e[q].x + __popc(e[q].y & (bit[q] - 1u));
      src[q] = (pidx<L::nQ>(q, j) & m) | (pidx<L::nQ>(L::rev(q), i) & ~m);
    }
  }
};

// PZ: the box is periodic along the row axis.
template <bool PZ>
struct WinWrap {};
template <>
struct WinWrap<true> {
  const uint32_t* __restrict__ count;  // fluid cells of each padded row
  int32_t EZ;                          // cells per row
};
template <bool PZ>
struct RowWinT : WinWrap<PZ> {
  static constexpr bool kOff32 = true, kOrdered = true;
  const uint32_t* __restrict__ coord;  // X << 22 | Y << 12 | Z
  const uint32_t* __restrict__ win;    // fluid bits << kWinBase | base, per (padded row, word)
  const uint32_t* __restrict__ plane;  // first node of each padded X; null: the bases count from node 0
  int32_t PY;  // padded rows along Y: E_Y + 2
  int32_t W;   // words per row (win_words)
  const int32_t* __restrict__ order = nullptr;  // block order, or null

  // What a node reads of its 9 (D3Q19) or 3 (D2Q9) neighbouring rows: the
  // words, and the index of the first fluid cell at or after z.
  template <class L>
  struct Rows {
    static constexpr int NY = L::nD == 3 ? 3 : 1;
    uint32_t b0[3 * NY], m[3 * NY];
    uint32_t t;  // bit of cell z - 1
    // PZ: what to add for a source at z - 1 (z = 0) and to take away for one
    // at z + 1 (z = E_Z - 1): the row's fluid cells, else 0
    uint32_t lo[3 * NY], hi[3 * NY];
    // row, step along z and fluid mask (all ones or zero) of the source cell r - c_q
    __device__ __forceinline__ static constexpr int row(int q) {
      return (1 - cx<L>(q)) * NY + (NY > 1 ? 1 - cy<L>(q) : 0);
    }
    // row k has sources at z - 1 and z + 1 (the rows along x = y hold only c_z = 0)
    __device__ __forceinline__ static constexpr bool off_z(int k) { return NY == 1 || k / NY == 1 || k % NY == 1; }
    __device__ __forceinline__ uint32_t fluid(int q) const {
      return static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int32_t>(m[row(q)]), t + 1 - cz<L>(q), 1));
    }
    // compact index of the source cell, where it is fluid
    __device__ __forceinline__ uint32_t node(int q) const {
      const int k = row(q), dz = -cz<L>(q);
      if (dz == 0) return b0[k];
      if (dz < 0) return PZ ? b0[k] - 1u + lo[k] : b0[k] - 1u;
      const uint32_t j = b0[k] + ((m[k] >> (t + 1u)) & 1u);
      return PZ ? j - hi[k] : j;
    }
  };

  // The window table is indexed by the halo-padded row (X+1, Y+1): halo rows
  // of a periodic axis repeat the rows they wrap to, those of a closed axis
  // are empty (all solid).  The neighbouring rows of a node are then one
  // vector offset plus a per-direction uniform base.
  template <class L>
  __device__ __forceinline__ void rows(int32_t i, Rows<L>& r) const {
    cell_rows<L>(coord[i], r);
  }
  template <class L>
  __device__ __forceinline__ void cell_rows(uint32_t c, Rows<L>& r) const {
    const uint32_t X = c >> 22, Y = (c >> 12) & 1023u, Z = c & 4095u;
    r.t = kWinBase + (Z & (kWinCells - 1u));
    const uint32_t pr = (X + 1u) * static_cast<uint32_t>(PY) + (Y + 1u);
    const uint32_t at = pr * static_cast<uint32_t>(W) + (Z >> kWinLog);
    constexpr int NY = Rows<L>::NY;
#pragma unroll
    for (int k = 0; k < 3 * NY; ++k) {
      const int dx = k / NY - 1, dy = NY > 1 ? k % NY - 1 : 0;
      r.m[k] = ld32(win + (dx * PY + dy) * W, at);
    }
    uint32_t first[3] = {0u, 0u, 0u};
    if (plane) {
#pragma unroll
      for (int d = 0; d < 3; ++d) first[d] = ld32(plane + d, X);
    }
    if constexpr (PZ) {
      const uint32_t last = static_cast<uint32_t>(this->EZ) - 1u;
#pragma unroll
      for (int k = 0; k < 3 * NY; ++k) r.lo[k] = r.hi[k] = 0u;
      if (Z == 0u || Z == last) {
#pragma unroll
        for (int k = 0; k < 3 * NY; ++k) {
          if (!Rows<L>::off_z(k)) continue;
          const int dx = k / NY - 1, dy = NY > 1 ? k % NY - 1 : 0;
          const uint32_t n = ld32(this->count + (dx * PY + dy), pr);
          r.lo[k] = Z == 0u ? n : 0u;
          r.hi[k] = Z == last ? n : 0u;
        }
      }
    }
    const uint32_t below = (2u << r.t) - (2u << kWinBase);  // cells of the word before z
#pragma unroll
    for (int k = 0; k < 3 * NY; ++k)
      r.b0[k] = (r.m[k] & ((1u << kWinBase) - 1u)) + (static_cast<uint32_t>(__popc(r.m[k] & below)) + first[k / NY]);
  }

  template <class L>
  __device__ __forceinline__ void sources(int32_t i, uint32_t (&src)[L::nQ - 1]) const {
    Rows<L> r;
    rows<L>(i, r);
    row_sources<L>(i, r, src);
  }
  template <class L>
  __device__ __forceinline__ static void row_sources(int32_t i, const Rows<L>& r, uint32_t (&src)[L::nQ - 1]) {
#pragma unroll
    for (int q = 0; q < L::nQ - 1; ++q) {
      // both candidates, combined by a mask: a per-lane select, not a branch
      const uint32_t m = r.fluid(q);
      src[q] = (pidx<L::nQ>(q, r.node(q)) & m) | (pidx<L::nQ>(L::rev(q), i) & ~m);
    }
  }

  // element at a 32-bit byte offset from a uniform base (tables below 4 GiB)
  __device__ __forceinline__ static uint32_t ld32(const uint32_t* __restrict__ p, uint32_t e) {
    return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(p) + e * 4u);
  }
};
using RowWin = RowWinT<false>;
using RowWinZ = RowWinT<true>;

// A pointer kept in memory, read as one into device memory: its accesses are
// then global instructions (scalar base, 32-bit offset) instead of flat ones
// with 64-bit address arithmetic per lane (batched FP32S step: 487 VALU
// instructions per wave for 602; 24 solves of 32^3 to 128^3, with descriptors
// read by scalar loads and items in XCD order: 88 us per step for 104, two-phase
// collision 87 for 93, colour 48 for 53).
template <typename T>
__host__ __device__ __forceinline__ T* device_ptr(T* const& p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(1))) T G;
  return (T*)*reinterpret_cast<G* const*>(&p);
#else
  return p;
#endif
}

// Windows of a batched solve.
__host__ __device__ __forceinline__ RowWin solve_windows(const BatchSolve& s) {
  return RowWin{{}, device_ptr(s.coord), device_ptr(s.win), device_ptr(s.plane), s.PY, s.W, nullptr};
}

// Work items of a batched launch.  Positions p = blockIdx, blockIdx + grid, ...
// name NS items each (one per 256-thread slice sub of the workgroup); items 8
// apart belong to one XCD's run (interleave_xcds), and the grid is a multiple
// of 8 wherever a workgroup takes more than one position.
template <int NS>
__host__ __device__ __forceinline__ int32_t batch_positions(int32_t n_items) {
  return NS == 1 ? n_items : (n_items + 8 * NS - 1) / (8 * NS) * 8;
}
// the item at it, known to be the same for the wave: its solve's descriptor is
// then read with scalar loads
__device__ __forceinline__ uint32_t wave_item(const uint32_t* __restrict__ items, int32_t it) {
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int32_t>(items[it])));
}
template <int NS>
__device__ __forceinline__ int32_t batch_item(int32_t p, int32_t sub) {
  return NS == 1 ? p : (p >> 3) * (8 * NS) + 8 * sub + (p & 7);
}

// The source node of every direction: bit q of fluid is set when the source
// cell of direction q is the fluid node j[q] (else a solid, and j[q] is
// undefined).
template <class L, bool PZ>
__device__ __forceinline__ void rowwin_links(const RowWinT<PZ>& ad, int32_t i, uint32_t (&j)[L::nQ - 1],
                                             uint32_t& fluid) {
  typename RowWinT<PZ>::template Rows<L> r;
  ad.template rows<L>(i, r);
  fluid = 0u;
#pragma unroll
  for (int q = 0; q < L::nQ - 1; ++q) {
    fluid |= r.fluid(q) & (1u << q);
    j[q] = r.node(q);
  }
}

// Colour of the neighbours neighbor(qq, n) for the colour gradient
// (LButilities.h:12-22): a fluid neighbour's phi; a solid neighbour's wall
// colour, per wall slot with the link table or one value for the whole node
// list with the row windows; 0 for the ghost node 0.  pn[Q-1] = 0.
struct WallPhi {
  const double* slot;  // per wall slot (link table)
  double uniform;      // every solid neighbour (row windows)
};

template <class L, typename T>
__device__ __forceinline__ void neighbour_phi(const TableAddr& ad, int32_t i, const T* __restrict__ phi,
                                              const WallPhi& wp, T (&pn)[L::nQ]) {
#pragma unroll
  for (int qq = 0; qq < L::nQ - 1; ++qq) {
    const int q = L::rev(qq);  // neighbor(qq, n) is the stream source of rev(qq)
    const uint32_t l = ad.link[static_cast<uint32_t>(q) * ad.NP + i];
    const uint32_t kind = l >> 30;
    const uint32_t j = l & kLinkIndexMask;
    pn[qq] = kind == kLinkStream ? phi[j] : (kind == kLinkBounce ? static_cast<T>(wp.slot[j]) : static_cast<T>(0));
  }
  pn[L::nQ - 1] = static_cast<T>(0);
}

template <class L, typename T, bool PZ>
__device__ __forceinline__ void neighbour_phi(const RowWinT<PZ>& ad, int32_t i, const T* __restrict__ phi,
                                              const WallPhi& wp, T (&pn)[L::nQ]) {
  uint32_t j[L::nQ - 1], fluid;
  rowwin_links<L>(ad, i, j, fluid);
  const T pw = static_cast<T>(wp.uniform);
#pragma unroll
  for (int qq = 0; qq < L::nQ - 1; ++qq) {
    const int q = L::rev(qq);
    // load from the node itself where the neighbour is solid (always in
    // bounds), then select: no branch
    const bool f = (fluid >> q) & 1u;
    const T v = phi[f ? j[q] : static_cast<uint32_t>(i)];
    pn[qq] = f ? v : pw;
  }
  pn[L::nQ - 1] = static_cast<T>(0);
}

// Element access of a population buffer: 32-bit byte offsets from the base
// when the layout guarantees the buffer is below 4 GiB (global loads with a
// scalar base and a 32-bit vector offset), 64-bit addresses otherwise.
template <bool OFF32, typename T>
__device__ __forceinline__ T ld_elem(const T* __restrict__ base, uint32_t e) {
  if (OFF32) return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + e * static_cast<uint32_t>(sizeof(T)));
  return base[e];
}
// Store of a population.  NT (streaming): the line leaves the L2 and takes no
// place in the MALL, for buffers that the MALL does not hold anyway; else the
// next step finds it there (stream_stores in layout_select.hpp).
template <bool NT, typename T>
__device__ __forceinline__ void st_elem(T v, T* p) {
  if (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}
template <bool OFF32, typename T>
__device__ __forceinline__ T* elem_ptr(T* __restrict__ base, uint32_t e) {
  if (OFF32) return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + e * static_cast<uint32_t>(sizeof(T)));
  return base + e;
}

}  // namespace lbamd
