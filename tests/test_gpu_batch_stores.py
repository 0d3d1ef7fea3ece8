"""A batch whose populations together fill more than the L2s but less than the
MALL writes with plain stores, a smaller one and a larger one with streaming
stores: the same k on every route, and that of a context of its own."""
import numpy as np
import pytest

import lbamd

pytestmark = pytest.mark.gpu

TAU, FORCE = 1.0, (1e-6, 0.0, 0.0)


def run(geos, precision, rho0=None):
    b = lbamd.Batch(lbamd.D3Q19, precision, 1 << 32, 50)
    for i, g in enumerate(geos):
        if rho0 is None:
            assert b.add(g, "x", TAU, FORCE, 1e-30, 100, i)
        else:
            assert b.add_twophase(g, "x", rho0[i], 1.0, 1.0, 0.8, 0.01, 0.7, FORCE, 1e-30, 100, i)
    out = {}
    while len(out) < len(geos):
        b.advance(1)
        for r in b.collect():
            out[r["tag"]] = (r["k"], tuple(r["k_phase"]), r["steps"])
    b.close()
    return [out[i] for i in range(len(geos))]


@pytest.mark.parametrize("two_phase", [False, True])
@pytest.mark.parametrize("precision", [lbamd.FP64, lbamd.FP32S, lbamd.FP16S])
def test_store_routes_agree(gpu_available, precision, two_phase):
    # 96^3 at porosity 0.5 has 0.44 M nodes: 34 MB (FP16S) to 134 MB (FP64) per
    # field of both buffers, 32^3 a 27th of that; six of the large ones in FP64
    # and FP32S pass 256 MB.
    big = lbamd.sphere_pack((96, 96, 96), 9.0, 0.5, 1, periodic="x", walls=True)[0]
    small = lbamd.sphere_pack((32, 33, 31), 4.0, 0.45, 2, periodic="x", walls=True)[0]
    rng = np.random.default_rng(3)
    rho = (lambda g: rng.random(g.shape)) if two_phase else None
    rb, rs = (rho(big), rho(small)) if two_phase else (None, None)
    alone = run([small], precision, two_phase and [rs] or None)[0]      # streaming: below 20 MB
    mid = run([big, small], precision, two_phase and [rb, rs] or None)  # plain below 256 MiB
    many = run([big] * 6 + [small], precision, two_phase and [rb] * 6 + [rs] or None)
    assert mid[1] == alone == many[6]
    assert all(m == mid[0] for m in many[:6])


@pytest.mark.parametrize("precision", [lbamd.FP64, lbamd.FP32S, lbamd.FP16S])
def test_store_routes_equal_contexts(gpu_available, precision):
    """Solves of a batch that writes with plain stores against a context for each."""
    geos = [lbamd.sphere_pack(n, r, p, s, periodic="x", walls=True)[0]
            for n, r, p, s in (((96, 96, 96), 9.0, 0.5, 1), ((32, 33, 31), 4.0, 0.45, 2))]
    for geo, got in zip(geos, run(geos, precision)):
        topo = lbamd.Topology.from_geometry(geo, lbamd.D3Q19, "x")
        ctx = lbamd.Context(lbamd.D3Q19, precision)
        ctx.set_topology_from(topo)
        ctx.init_equilibrium(1, 0, np.ones(topo.n_nodes), np.zeros((topo.n_nodes, 3)))
        k, steps = ctx.solve_permeability(TAU, FORCE, 50, 1e-30, 100, float(geo.size))
        ctx.close()
        topo.close()
        assert (got[0], got[2]) == (k, steps)
