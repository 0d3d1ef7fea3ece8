"""Field downloads of several contexts at the same time, one thread each: they
share the process's pinned stages (csrc/capi.hip), small and large ones in turn,
and every download gets its own context's values."""
import threading

import numpy as np
import pytest

import lbamd

pytestmark = pytest.mark.gpu


def test_downloads_on_threads(gpu_available):
    sizes = [(20, 18, 33), (64, 50, 60), (150, 140, 130), (24, 30, 28), (90, 80, 70), (40, 41, 42)]
    ctxs, want = [], []
    for n, size in enumerate(sizes):
        geo, _ = lbamd.sphere_pack(size, 4.0, 0.55, n + 1, periodic="x", walls=True)
        topo = lbamd.Topology.from_geometry(geo, lbamd.D3Q19, "x")
        ctx = lbamd.Context(lbamd.D3Q19, lbamd.FP64)
        ctx.set_topology_from(topo)
        rng = np.random.default_rng(n)
        ctx.init_equilibrium(1, 0, 1.0 + 1e-2 * rng.random(topo.n_nodes), np.zeros((topo.n_nodes, 3)))
        ctx.step_bgk(3, 0.9, (1e-5, 0.0, 0.0))
        topo.close()
        ctxs.append(ctx)
        want.append((ctx.download_scalar(lbamd.RHO), ctx.download_vel()))
    assert 24 * np.count_nonzero(want[2][0]) > 32 << 20  # more than a stage: in parts
    bad = []

    def work(n):
        for _ in range(25):
            if not (np.array_equal(ctxs[n].download_scalar(lbamd.RHO), want[n][0])
                    and np.array_equal(ctxs[n].download_vel(), want[n][1])):
                bad.append(n)

    threads = [threading.Thread(target=work, args=(n,)) for n in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for ctx in ctxs:
        ctx.close()
    assert not bad, bad
