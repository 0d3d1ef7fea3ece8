// Contexts where pinned host memory is short, or graphs cannot be made.  The
// program's own hipHostMalloc and hipGraphInstantiate stand before the runtime's:
// they count the calls and, with "nopin" or "nograph", refuse them.  argv: pin |
// nopin | nograph, output file (every downloaded value and solve, as doubles),
// and the memory of the halo buffers: pageable | pinned | device | managed.
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "badchimp_amd.h"

static int pins = 0, graphs = 0;
static bool refuse = false, refuse_graphs = false;
extern "C" int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  using Malloc = int (*)(void**, size_t, unsigned);
  static const Malloc next = reinterpret_cast<Malloc>(dlsym(RTLD_NEXT, "hipHostMalloc"));
  ++pins;
  return refuse ? 2 /* hipErrorOutOfMemory */ : next(p, bytes, flags);
}

extern "C" int hipGraphInstantiate(void** exec, void* graph, void** node, char* log, size_t bytes) {
  using Instantiate = int (*)(void**, void*, void**, char*, size_t);
  static const Instantiate next = reinterpret_cast<Instantiate>(dlsym(RTLD_NEXT, "hipGraphInstantiate"));
  ++graphs;
  return refuse_graphs ? 2 : next(exec, graph, node, log, bytes);
}

extern "C" {
int hipMalloc(void**, size_t);
int hipMallocManaged(void**, size_t, unsigned);
int hipMemcpy(void*, const void*, size_t, int);
int hipFree(void*);
int hipHostFree(void*);
}

static lb_ctx* ctx = nullptr;
static void ok(int rc, const char* what) {
  if (rc == LB_OK) return;
  std::printf("%s: %d %s\n", what, rc, lb_last_error(ctx));
  std::exit(1);
}
static std::vector<double> all;
static void keep(const std::vector<double>& v) { all.insert(all.end(), v.begin(), v.end()); }

// a halo buffer of n doubles in the memory asked for
struct Buffer {
  char kind;  // second letter: a(geable), i(nned), e(vice), managed as M
  size_t n;
  double* p = nullptr;
  Buffer(const char* name, size_t count) : kind(*name == 'm' ? 'M' : name[1]), n(count) {
    void** q = reinterpret_cast<void**>(&p);
    const int e = kind == 'e' ? hipMalloc(q, n * 8) : kind == 'M' ? hipMallocManaged(q, n * 8, 1)
                  : kind == 'i' ? hipHostMalloc(q, n * 8, 0) : (*q = std::calloc(n, 8)) == nullptr;
    if (e != 0) {
      std::printf("%s buffer: %d\n", name, e);
      std::exit(1);
    }
  }
  ~Buffer() {
    if (kind == 'e' || kind == 'M') (void)hipFree(p);
    else if (kind == 'i') (void)hipHostFree(p);
    else std::free(p);
  }
  void set(const std::vector<double>& v) { ok(hipMemcpy(p, v.data(), v.size() * 8, 4), "copy in"); }
  std::vector<double> get(size_t count) const {
    std::vector<double> v(count);
    ok(hipMemcpy(v.data(), p, count * 8, 4), "copy out");
    return v;
  }
};

struct Lists {
  int32_t n = 0;
  std::vector<int32_t> nb, pos, bulk;
  std::vector<int16_t> types;
};
static Lists lists(const int32_t* dims, const std::vector<int32_t>& geo, int rank) {
  lb_topo* t = nullptr;
  ok(lb_topo_from_geometry(LB_D3Q19, 3, dims, geo.data(), 1, rank, &t), "geometry");
  Lists l;
  l.n = lb_topo_num_nodes(t);
  l.nb.resize(static_cast<size_t>(l.n) * 19);
  l.pos.resize(static_cast<size_t>(l.n) * 3);
  l.types.resize(l.n);
  l.bulk.resize(lb_topo_num_bulk(t));
  ok(lb_topo_neighbors(t, l.nb.data()), "neighbours");
  ok(lb_topo_positions(t, l.pos.data()), "positions");
  ok(lb_topo_node_types(t, l.types.data()), "types");
  ok(lb_topo_bulk(t, l.bulk.data()), "bulk");
  lb_topo_destroy(t);
  return l;
}
static void set(const Lists& l, int precision) {
  ok(lb_ctx_create(LB_D3Q19, precision, 0, &ctx), "context");
  ok(lb_set_topology_grid(ctx, l.n, l.nb.data(), l.types.data(), l.bulk.data(), static_cast<int32_t>(l.bulk.size()),
                          l.pos.data(), 0),
     "topology");
}
static void fields(int n, int nf) {
  std::vector<double> rho(static_cast<size_t>(n) * nf), vel(static_cast<size_t>(n) * 3), phi(n);
  ok(lb_download_scalar(ctx, LB_RHO, nf, rho.data()), "density");
  ok(lb_download_vector(ctx, LB_VEL, 1, vel.data()), "velocity");
  keep(rho);
  keep(vel);
  if (nf == 2) {
    ok(lb_download_scalar(ctx, LB_PHI, 1, phi.data()), "colour");
    keep(phi);
  }
}

int main(int argc, char** argv) {
  if (argc != 4) return 2;
  refuse = !std::strcmp(argv[1], "nopin");
  refuse_graphs = !std::strcmp(argv[1], "nograph");
  const int32_t dims[3] = {20, 18, 33};
  std::vector<int32_t> geo(20 * 18 * 33), split;
  uint32_t r = 7;
  for (size_t k = 0; k < geo.size(); ++k) {
    const size_t y = k / 33 % 18, z = k % 33;
    r = r * 1664525u + 1013904223u;
    geo[k] = y != 0 && y != 17 && z != 0 && z != 32 && r >> 30 != 0;
  }
  const double force[3] = {1e-4, 2e-5, 0.0};
  const Lists whole = lists(dims, geo, 1);
  std::vector<double> rho(static_cast<size_t>(whole.n) * 2), rest(static_cast<size_t>(whole.n) * 3, 0.0);
  for (int32_t k = 0; k < whole.n; ++k) {
    rho[2 * k] = 0.2 + 0.01 * (k % 60);
    rho[2 * k + 1] = 1.0 - rho[2 * k];
  }
  // one field in FP64, two in float storage
  set(whole, LB_FP64);
  ok(lb_init_equilibrium(ctx, 1, 0, 2, 0, rho.data(), rest.data()), "initial state");
  ok(lb_step_bgk(ctx, 7, 0.9, force), "steps");
  std::printf("pinned before a download %d\n", pins);
  fields(whole.n, 1);
  lb_ctx* const one = ctx;
  set(whole, LB_FP32S);
  ok(lb_set_wall_densities(ctx, rho.data()), "wall densities");
  for (int k = 0; k < 2; ++k) ok(lb_init_equilibrium(ctx, 2, k, 2, k, rho.data(), rest.data()), "initial state");
  ok(lb_step_cg(ctx, 5, 0.9, 1.1, 0.01, 0.7, LB_FORCE_FIXED, force), "two-phase steps");
  fields(whole.n, 2);
  lb_ctx_destroy(ctx);
  ctx = one;
  fields(whole.n, 1);
  lb_ctx_destroy(ctx);
  std::printf("pinned for fields %d\n", pins);
  // a rank of a split domain with one exchange: what it packs, and its fields
  // and colour after an unpack
  split = geo;
  for (size_t k = split.size() / 2; k < split.size(); ++k) split[k] *= 2;
  const Lists part = lists(dims, split, 1);
  std::vector<int32_t> send(part.bulk.begin(), part.bulk.begin() + 50), recv;
  for (int32_t k = 1; k < part.n; ++k)
    if (part.types[k] == 4) recv.push_back(k);
  const int32_t ns = static_cast<int32_t>(send.size()), nr = static_cast<int32_t>(recv.size());
  const std::vector<int32_t> two(send.size(), 2), one_dir(recv.size(), 1), dir(recv.size(), 3);
  std::vector<int32_t> dirs;
  for (int32_t k = 0; k < ns; ++k) dirs.insert(dirs.end(), {0, 4});
  Buffer out(argv[3], 4 * send.size()), in(argv[3], 2 * recv.size());
  std::vector<double> got(2 * recv.size());
  for (size_t k = 0; k < got.size(); ++k) got[k] = 0.01 + 1e-4 * static_cast<double>(k % 17);
  in.set(got);
  for (int nf = 1; nf <= 2; ++nf) {
    int32_t x = -1;
    set(part, LB_FP64);
    ok(lb_set_wall_densities(ctx, rho.data()), "wall densities");
    ok(lb_halo_add(ctx, 1, ns, send.data(), two.data(), dirs.data(), nr, recv.data(), one_dir.data(), dir.data(), &x),
       "exchange");
    for (int k = 0; k < nf; ++k) ok(lb_init_equilibrium(ctx, nf, k, 2, k, rho.data(), rest.data()), "initial state");
    for (int s = 0; s < 3; ++s) {
      if (nf == 1) {
        ok(lb_step_bgk(ctx, 1, 0.9, force), "step");
      } else {
        ok(lb_step_cg_colour(ctx, nullptr), "colour");
        ok(lb_halo_pack_colour(ctx, x, out.p), "pack colour");
        keep(out.get(ns));
        ok(lb_halo_unpack_colour(ctx, x, in.p), "unpack colour");
        ok(lb_step_cg_collide(ctx, 0.9, 1.1, 0.01, 0.7, LB_FORCE_FIXED, force, 0.0), "collision");
      }
      ok(lb_halo_pack(ctx, x, nf, out.p), "pack");
      keep(out.get(2 * ns * nf));
      ok(lb_halo_unpack(ctx, x, nf, in.p), "unpack");
    }
    fields(part.n, nf);
    lb_ctx_destroy(ctx);
  }
  // a solve whose steps replay graphs
  set(whole, LB_FP32S);
  ok(lb_init_equilibrium(ctx, 1, 0, 2, 0, rho.data(), rest.data()), "initial state");
  double k = 0.0;
  int64_t steps = 0;
  graphs = 0;
  ok(lb_solve_permeability(ctx, 0.9, force, 101, 1e-30, 606, 20.0 * 18 * 33, &k, &steps), "solve");
  keep({k, static_cast<double>(steps)});
  std::printf("graphs %d\n", graphs);
  fields(whole.n, 1);
  lb_ctx_destroy(ctx);
  std::FILE* f = std::fopen(argv[2], "wb");
  if (!f || std::fwrite(all.data(), sizeof(double), all.size(), f) != all.size() || std::fclose(f)) return 1;
  std::printf("pinned %d, %zu values\n", pins, all.size());
  return 0;
}
