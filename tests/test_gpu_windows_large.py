"""Row windows of boxes that are periodic along the row axis, and windows whose
bases count from each x plane (node lists of 2^22 nodes and more), at sizes that
reach what small boxes do not: plain stores, the plane-by-plane block order and
the plane bases themselves, in contexts and in a batch.  Against the link table
of the same context, bit for bit; fluxes, whose terms the two layouts add in
another order, within 64 rounding steps of the sum of the absolute terms; a
batched solve against the same solve of a context."""
import numpy as np
import pytest

import lbamd

pytestmark = pytest.mark.gpu

F = (1e-4, 1e-5, -2e-5)
EPS = np.finfo(float).eps


def solids(shape, share, periodic, seed):
    geo = (np.random.default_rng(seed).random(shape) >= share).astype(np.int32)
    for a, name in enumerate("xyz"):
        if name not in periodic:
            idx = [slice(None)] * 3
            idx[a] = [0, -1]
            geo[tuple(idx)] = 0
    return geo


def context(topo, precision, table, two_phase):
    ctx = lbamd.Context(lbamd.D3Q19, precision)
    ctx.set_topology_from(topo, table_only=table)
    rng = np.random.default_rng(4)
    vel = 1e-2 * rng.standard_normal((topo.n_nodes, 3))
    if two_phase:
        r0 = rng.random(topo.n_nodes)
        rho = np.stack([r0, 1.0 - r0], axis=-1)
        rho[topo.node_types() == 1] = (0.8, 0.2)
        ctx.set_wall_densities(rho)
        for k in range(2):
            ctx.init_equilibrium(2, k, rho, vel, rho_field=k)
    else:
        ctx.init_equilibrium(1, 0, 1.0 + 1e-2 * rng.standard_normal(topo.n_nodes), vel)
    return ctx


def steps(ctx, n, op):
    if op == "cg":
        ctx.step_cg(n, 0.9, 1.1, 0.01, 0.7, lbamd.FORCE_FIXED, F)
    elif op == "trt":
        ctx.step_trt(n, 1.0, 0.875, F)
    else:
        ctx.step_bgk(n, 0.9, F)


def same(topo, precision, op, z_periodic, chunks, populations=True):
    nf, b = (2 if op == "cg" else 1), topo.bulk()
    out = []
    for table in (False, True):
        ctx = context(topo, precision, table, nf == 2)
        note = "rows (periodic along the row axis)" if z_periodic else "row windows"
        assert table or ctx.layout_note == note, ctx.layout_note
        for n in chunks:
            steps(ctx, n, op)
        r = [ctx.download_scalar(lbamd.RHO, nf)[b], ctx.download_vel()[b]]
        if nf == 2:
            r.append(ctx.download_scalar(lbamd.PHI)[b])
        flux = [np.array(ctx.reduce_flux(d)) for d in range(3)]
        if populations:
            r.append(ctx.download_f(nf)[b])
        ctx.close()
        out.append((r, flux))
    (win, fw), (tab, ft) = out
    for x, y in zip(win, tab):
        assert np.isfinite(x).all() and np.array_equal(x, y)
    # sum_n sum_q |f_q c_q| <= sum_n rho_n
    bound = 64 * EPS * np.abs(win[0]).sum()
    for x, y in zip(fw, ft):
        assert np.abs(x - y).max() <= bound, (x, y, bound)


@pytest.mark.parametrize("op", ["bgk", "trt", "cg"])
@pytest.mark.parametrize("precision", [lbamd.FP64, lbamd.FP32S])
def test_periodic_rows_above_the_l2(gpu_available, precision, op):
    """0.33 M nodes, 18 blocks per x plane: 25 MB (FP32S, one field) to 200 MB of populations."""
    topo = lbamd.Topology.from_geometry(solids((70, 83, 85), 0.33, "xyz", 5), lbamd.D3Q19, "xyz")
    assert topo.n_bulk > 8 * 256 * 70
    same(topo, precision, op, True, (1, 2, 9))
    topo.close()


@pytest.mark.parametrize("periodic,op", [("xyz", "bgk"), ("xz", "cg"), ("xy", "cg")])
def test_plane_bases(gpu_available, periodic, op):
    geo = solids((112, 205, 207), 0.08, periodic, 6)
    topo = lbamd.Topology.from_geometry(geo, lbamd.D3Q19, periodic)
    assert topo.n_bulk >= 1 << 22
    same(topo, lbamd.FP32S, op, "z" in periodic, (3,), populations=False)
    topo.close()


@pytest.mark.parametrize("two_phase", [False, True])
def test_plane_bases_in_a_batch(gpu_available, two_phase):
    geo = solids((112, 207, 209), 0.08, "x", 7)
    small = solids((24, 20, 28), 0.4, "x", 8)
    force = (1e-6, 0.0, 0.0)
    topo = lbamd.Topology.from_geometry(geo, lbamd.D3Q19, "x")
    assert topo.n_bulk >= 1 << 22
    ctx = lbamd.Context(lbamd.D3Q19, lbamd.FP32S)
    ctx.set_topology_from(topo)
    if two_phase:
        sw = (np.random.default_rng(9).random(geo.shape) < 0.5) * (geo > 0) * 1.0
        rho, pos = np.zeros((topo.n_nodes, 2)), topo.positions()
        fluid = topo.bulk()
        rho[fluid, 0] = sw[tuple(np.mod(pos[fluid], geo.shape).T)]
        rho[fluid, 1] = 1.0 - rho[fluid, 0]
        rho[topo.node_types() == 1] = (1.0, 0.0)
        ctx.set_wall_densities(rho)
        # both fields at once, as the batch stores its rest state (two calls of
        # init_equilibrium round the first field twice in float storage)
        w = np.array([2.0] * 3 + [1.0] * 6 + [2.0] * 3 + [1.0] * 6 + [12.0]) / 36.0
        ctx.upload_f(w * rho[:, :, None])
        k, n = ctx.solve_relperm(0.9, 1.1, 0.01, 0.7, force, 5, 1e-30, 10, float(geo.size))
    else:
        ctx.init_equilibrium(1, 0, np.ones(topo.n_nodes), np.zeros((topo.n_nodes, 3)))
        k, n = ctx.solve_permeability(1.0, force, 5, 1e-30, 10, float(geo.size))
    ctx.close()
    topo.close()
    b = lbamd.Batch(lbamd.D3Q19, lbamd.FP32S, 4 << 30, 5)
    assert b.add(small, "x", 1.0, force, 1e-30, 10, 0)
    if two_phase:
        assert b.add_twophase(geo, "x", sw, 1.0, 0.9, 1.1, 0.01, 0.7, force, 1e-30, 10, 1)
    else:
        assert b.add(geo, "x", 1.0, force, 1e-30, 10, 1)
    got = {}
    while len(got) < 2:
        b.advance(1)
        for r in b.collect():
            got[r["tag"]] = r
    b.close()
    assert got[1]["steps"] == n == 10
    if two_phase:
        assert np.all(np.isfinite(k)) and np.array_equal(got[1]["k_phase"], k), (got[1], k)
    else:
        assert np.isfinite(k) and k > 0 and got[1]["k"] == k, (got[1], k)
