"""Row windows (csrc/addressing.hpp, csrc/rowbuild.hpp) against the geometry.

For boxes whose rows end inside a window word, at its end and one cell after
it, with every combination of periodic axes, each fluid cell's neighbours as
the windows give them (the host restatement that every context checks its
links with) must be the cells of the box: solid, or the compact index in row
order.  The bases count from node 0 and from the first node of each x plane,
the form that node lists above 2^22 nodes take."""
import os
import subprocess

import pytest

import lbamd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include "rowbuild.hpp"
#include <cstdio>
#include <map>
#include <random>
using namespace lbamd;
static int fails = 0;
static void box(int lattice, const int32_t* d, int mask, unsigned seed) {
  const int nD = lattice == LB_D2Q9 ? 2 : 3;
  int64_t n = 1;
  for (int a = 0; a < nD; ++a) n *= d[a];
  std::mt19937 r(seed);
  std::vector<int32_t> geo(n);
  for (auto& g : geo) g = r() % 10 < 6;
  geo[n / 2] = 1;
  RowBuild rb;
  std::string why;
  if (!rows_from_geometry(lattice, d, geo.data(), mask, rb, why)) { std::printf("rows: %s\n", why.c_str()); ++fails; return; }
  std::map<uint32_t, int64_t> at;  // packed cell -> compact index
  for (size_t i = 0; i < rb.coord.size(); ++i) at[rb.coord[i]] = static_cast<int64_t>(i);
  for (int planes = 0; planes < 2; ++planes) {
    WinBuild wb;
    if (!build_windows(rb, true, wb, why, planes != 0)) { std::printf("windows: %s\n", why.c_str()); ++fails; return; }
    if ((planes != 0) == wb.plane.empty() || ((rb.g.periodic & 4) != 0) == wb.count.empty()) ++fails;
    const int Q = lattice == LB_D2Q9 ? 9 : 19;
    for (size_t i = 0; i < rb.coord.size(); ++i)
      for (int q = 0; q < Q - 1; ++q) {
        int32_t X[3] = {static_cast<int32_t>(rb.coord[i] >> 22), static_cast<int32_t>((rb.coord[i] >> 12) & 1023u),
                        static_cast<int32_t>(rb.coord[i] & 4095u)};
        bool in = true;
        for (int a = 0; a < 3; ++a) {
          X[a] -= lattice == LB_D2Q9 ? (a == 0 ? D2Q9::c(q, 0) : a == 2 ? D2Q9::c(q, 1) : 0) : D3Q19::c(q, a);
          in = RowGeom::wrap(X[a], rb.g.E[a], (rb.g.periodic >> a) & 1) && in;
        }
        const auto it = in ? at.find((uint32_t(X[0]) << 22) | (uint32_t(X[1]) << 12) | uint32_t(X[2])) : at.end();
        const auto s = win_source(lattice, rb, wb, q, static_cast<int32_t>(i));
        if (s.first != (it != at.end()) || (s.first && s.second != it->second)) ++fails;
      }
  }
}
int main() {
  unsigned seed = 1;
  for (int ez : {1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 40, 65})
    for (int ey : {2, 33})
      for (int mask = 0; mask < 8; ++mask) {
        const int32_t d3[3] = {5, ey, ez};
        box(LB_D3Q19, d3, mask, seed++);
        const int32_t d2[2] = {ey, ez};
        if (mask < 4) box(LB_D2Q9, d2, mask, seed++);
      }
  std::printf("fails %d\n", fails);
  return fails != 0;
}
'''


def test_windows_name_the_cells_of_the_box(tmp_path):
    src = tmp_path / "win.hip"
    src.write_text(SRC)
    exe = tmp_path / "win"
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "badchimp-cpp_amd", "csrc"), str(src), "-o", str(exe)], check=True,
                   capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and "fails 0" in out.stdout, out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("two_phase", [False, True])
@pytest.mark.parametrize("lattice,shape,periodic", [
    ("D3Q19", (9, 7, 2), "xyz"), ("D3Q19", (6, 35, 8), "xz"), ("D3Q19", (7, 6, 17), "xyz"),
    ("D3Q19", (5, 8, 40), "yz"), ("D3Q19", (8, 7, 9), "xy"), ("D2Q9", (11, 9), "xy"), ("D2Q9", (8, 16), "y"),
    ("D2Q9", (13, 25), "x")])
def test_windows_step_like_the_link_table(gpu_available, lattice, shape, periodic, two_phase):
    """Populations after 9 steps bit for bit, row windows against the link table (FP64)."""
    import numpy as np
    rng = np.random.default_rng(sum(shape))
    geo = (rng.random(shape) > 0.3).astype(np.int32)
    for a, name in enumerate("xyz"[: len(shape)]):
        if name not in periodic:  # closed axes get walls
            idx = [slice(None)] * len(shape)
            idx[a] = [0, -1]
            geo[tuple(idx)] = 0
    lat = lbamd.LATTICE_NAME[lattice]
    topo = lbamd.Topology.from_geometry(geo, lat, periodic)
    nf, Q = (2 if two_phase else 1), lbamd.Q_OF[lat]
    f0 = 1.0 / Q * (1.0 + 0.1 * rng.standard_normal((topo.n_nodes, nf, Q)))
    out = []
    for table in (False, True):
        ctx = lbamd.Context(lat, lbamd.FP64)
        ctx.set_topology_from(topo, table_only=table)
        z = "xyz"[len(shape) - 1] in periodic
        assert ctx.layout == (0 if table else 1 if z else 2)
        if z and not table:
            assert ctx.layout_note == "rows (periodic along the row axis)"
        if two_phase:
            ctx.set_wall_densities(np.tile([0.8, 0.2], (topo.n_nodes, 1)))
        ctx.upload_f(f0)
        for n in (1, 8):
            if two_phase:
                ctx.step_cg(n, 0.9, 1.1, 0.01, 0.7, lbamd.FORCE_FIXED, (1e-4, 1e-5, 0.0)[: len(shape)])
            else:
                ctx.step_bgk(n, 0.9, (1e-4, 1e-5, 0.0)[: len(shape)])
        b = topo.bulk()
        out.append((ctx.download_f(nf)[b], ctx.reduce_flux(0)))
        ctx.close()
    assert np.array_equal(out[0][0], out[1][0])
    if not two_phase:
        assert np.allclose(out[0][1], out[1][1], rtol=1e-12, atol=1e-13)
