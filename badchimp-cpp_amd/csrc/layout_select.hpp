// Which address layout a launch over some number of population fields uses.
//
// Pure host arithmetic (no HIP types), so that a CPU test can check the
// selection directly.
#pragma once
#include <cstdint>

namespace lbamd {

// Address layouts (addressing.hpp): link table, rows, row windows, and row
// windows of a box that is periodic along the row axis.
constexpr int kLayTable = 0, kLayRows = 1, kLayWin = 2, kLayWinZ = 3;

// The row windows address the population buffer with 32-bit byte offsets
// from its base, so every element of all n_fields fields of one buffer must
// lie below 4 GiB.
inline bool rowwin_fits(int Q, int64_t NP, int n_fields, int64_t elem_bytes) {
  return static_cast<uint64_t>(n_fields) * static_cast<uint64_t>(Q) * static_cast<uint64_t>(NP) *
             static_cast<uint64_t>(elem_bytes) <
         (1ull << 32);
}

// Whether the step kernels write populations with streaming stores, for both
// buffers of a context, or of all active solves of a batch, together.  While they
// fit the MALL's 256 MiB a plain store leaves the values where the next step reads
// them; beyond, a plain store only displaces lines that are still to be read.  Below
// 20 MB, where the buffers fit the L2s, a plain store is written back when the
// kernel ends, after its last node.  Plain / streaming, us per step:
// FP32S 64^3 pack (16 MB) 5.55 / 5.23, D2Q9 1021x509 (22 MB) 5.6 / 6.0, FP32S
// 80^3 (30 MB) 7.4 / 8.9, FP64 96^3 (107 MB) 19.3 / 23.7, FP16S 161x143x150
// (100 MB) 22.2 / 26.8, FP64 128^3 (255 MB) 40.4 / 47.6; two-phase FP64 64^3
// (62 MB) 22.0 / 22.0, 100^3 (245 MB) 59.1 / 62.4; beyond: FP32S 165^3 (273 MB)
// 52.9 / 50.9, FP64 256^3 366 / 351; around the limit FP64 128^3 periodic along all
// axes (255 MB) 46.6 / 49.5, FP32S 200x170x150 (265 MB) 53.5 / 50.7.  A batch of 4 packs of 64^3, FP32S (64 MB)
// 13.5 / 15.6, FP64 (128 MB) 22.6 / 26.8; 3 of 96^3, FP16S 20.6 / 24.7; 4 of
// 128^3, FP16S 56.1 / 67.4.
// The link table (link bytes, 0 for the other layouts) is read in every step and
// counts: FP32S 144^3 (177 MB and 84) 41.0 / 42.8, D2Q9 1000x4000 (202 and 90) 49.9 /
// 48.0, 160^3 (243 and 115) 66.3 / 61.3; FP64 112^3 (165 and 39) 35.9 / 38.3, 128^3
// (247 and 59) 56.4 / 54.7, 144^3 (353 and 84) 81.9 / 71.7; FP16S 160^3 (121 and 115)
// 41.4 / 43.1, 176^3 (162 and 153) 62.0 / 55.3.
// So do density and velocity (fields bytes) in calls of one or two steps, which all
// write them: FP32S 160^3 (243 MB and 51) 1 step per call 63.6 / 57.9, 2 55.9 / 53.1,
// 10 42.4 / 48.5; FP64 128^3 (247 and 26) 59.3 / 54.0, 51.0 / 50.8, 42.2 / 48.2; FP16S
// 200^3 (209 and 88) 77.9 / 73.7, 66.7 / 67.2, 50.9 / 58.6; within the limit FP64 120^3
// (203 and 22) 40.5 / 45.8, FP32S 150^3 (200 and 42) 42.4 / 48.6.
// Two fields, which the colour pass reads before the collision does: plain stores
// pay from 60 MB on only: FP32S D2Q9 800x400 (32 MB) 13.2 / 12.6,
// 800x600 (48 MB) 17.0 / 16.4, D3Q19 80^3 (59 MB) 20.1 / 19.9, 96^3 (103 MB) 32.9 /
// 34.2; FP64 64^3 (60 MB) 20.2 / 20.4, 80^3 (118 MB) 31.5 / 33.5; FP16S 80^3 (30 MB)
// 17.1 / 16.4, 112^3 (82 MB) 36.6 / 38.4; batches of two-phase solves, FP32S 3 of
// 48^3 (37 MB) 17.4 / 16.5, 6 (74 MB) 26.1 / 27.3, FP64 8 of 32^3 (56 MB) 21.4 /
// 21.8, 20 (140 MB) 39.4 / 43.0, FP16S 3 of 64^3 (45 MB) 25.9 / 25.6.  With the link table, which both passes
// read, they do not pay at all: FP32S 80^3 33.6 / 32.3, 112^3 (165 MB) 86.8 / 83.9, D2Q9
// 1000x1000 (101 MB) 43.6 / 42.1, FP64 96^3 (206 MB) 74.9 / 74.9; the exception is
// FP64 80^3 (118 MB) 42.9 / 43.9.
inline bool stream_stores(int64_t both_buffers, int n_fields = 1, int64_t link = 0, int64_t fields = 0) {
  if (n_fields == 2 && link > 0) return true;
  return both_buffers < (n_fields == 2 ? 60000000 : 20000000) || both_buffers + link + fields > 262000000;
}

// Whether the blocks of the row windows go to the XCDs plane by plane
// (block_order in rowbuild.hpp) or in runs of 4 (node_block), by the bytes of one
// population buffer and the storage form.  The plane order reads neighbouring rows
// from the XCD's own L2; its front is wider, eight runs of a plane, and from some
// size of the buffers on that costs more at the HBM than the L2 saves.  Plane
// order / runs, us per step, sphere packs of porosity 0.4 by MB per buffer:
// FP64    122 40.8 / 45.1, 291 105.2 / 106.8, 552 199.6 / 201.3, 635 226.1 /
//         229.2, 689 245.8 / 246.4; 725 263.2 / 260.3, 889 323.8 / 314.9, 1462
//         536.6 / 514.8, 2158 791.2 / 760.6; porosity 0.8, 817 281.7 / 279.8
// FP32S   276 105.6 / 107.6, 538 203.2 / 204.5, 602 230.0 / 231.6, 644 246.1 /
//         245.9; 731 279.4 / 274.1, 1079 415.0 / 404.8, 2073 828.2 / 783.7
// FP16S   644 342.3 / 342.2, 761 397.7 / 401.6; 892 466.5 / 463.3, 1036 548.6 / 535.0
// two fields, both of them counted:
// FP64    852 439 / 453, 1451 788.6 / 791.9, 2150 1171 / 1173; 3233 1802 / 1769,
//         3858 2160 / 2114
// FP32S   1075 627.4 / 635.9; 1462 857.7 / 854.2, 2158 1298 / 1272
// FP16S   1288 1033 / 1051, 1784 1421 / 1441 (larger ones not timed)
inline bool plane_order(int n_fields, int64_t elem_bytes, int64_t buffer) {
  if (n_fields == 1) return buffer <= (elem_bytes == 2 ? 820000000 : 700000000);
  return buffer <= (elem_bytes == 8 ? 2300000000 : elem_bytes == 4 ? 1350000000 : int64_t{1} << 32);
}

// Whether a D2Q9 list of n nodes takes kTileSteps steps per launch in tiles
// (tile2d.hpp) or one.  A tiled launch goes by its tiles, solid cells included, and
// costs another round of 256 workgroups (one more per CU) at a time: FP64 2.1 us per
// step up to 256 tiles, 2.9 up to 512, 3.65 up to 768, 4.4 up to 1024, 5.2 beyond.
// A plain step goes by its nodes: 3.2-3.6 us up to 256 blocks of 256 nodes, 4.0-4.5
// up to 512, 5.1 beyond.  So FP64 lists take tiles up to two rounds more than full
// rounds of blocks (less a few: 65 k nodes are 256 blocks).  Tiled / plain, BGK and
// TRT, us per step: 425 tiles, 29 k to 59 k nodes 2.80-3.20 / 3.40-3.66; 616 tiles,
// 66 k 3.65 / 3.96 and 3.79 / 3.99; 570, 62 k 3.72 / 3.67 and 3.80 / 3.68; 616, 42 k
// 3.70 / 3.48 and 3.89 / 3.50; 946, 130 k 4.44 / 4.72; 840, 94 k 4.51 / 4.26; 880,
// 60 k 4.38 / 3.67 and 4.59 / 3.70; 1100, 152 k 5.27 / 5.21.  Float storage, with half
// the LDS, pays up to 1000 tiles at every porosity from 0.5 on: 425 tiles 1.91-2.22
// / 3.08-3.20, 840 tiles, 59 k to 120 k nodes 2.96-3.22 / 3.12-3.54; beyond it depends
// on the solids: 1428 tiles, 198 k 3.71 / 4.57, 118 k 3.63 / 3.58, 2278 tiles, 190 k
// 4.96 / 4.33.
inline bool tiles_pay(int64_t elem_bytes, int64_t tiles, int64_t n) {
  if (elem_bytes == 4) return tiles <= 1000;
  const int64_t blocks = (n + 255) / 256;
  return (tiles + 255) / 256 <= 2 + (blocks + 8) / 256;
}

// Layout of a launch over n_fields fields: the context's layout, with the row
// windows replaced by the rows
// (64-bit addresses, same sources) when the fields do not fit below 4 GiB.
inline int launch_layout(int layout, int Q, int64_t NP, int n_fields, int64_t elem_bytes) {
  return layout >= kLayWin && !rowwin_fits(Q, NP, n_fields, elem_bytes) ? kLayRows : layout;
}

}  // namespace lbamd
