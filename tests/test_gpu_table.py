"""Viscosity tables around the size that a step keeps in LDS (256 rows with the
constant extension at both ends) against the oracle, FP64, bit for bit, and
FP32S norm-wise (velocity 1e-4, as in test_gpu_rheology.py)."""
import numpy as np
import pytest

import lbamd
import oracle
from helpers import OracleTopo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 2, 254, 255, 600])
@pytest.mark.parametrize("precision", [lbamd.FP64, lbamd.FP32S])
def test_table_sizes(gpu_available, rows, precision):
    rng = np.random.default_rng(rows)
    geo = (rng.random((9, 8, 7)) > 0.25).astype(np.int64)
    geo[:, 0] = geo[:, -1] = 0
    geo[:, :, 0] = geo[:, :, -1] = 0
    T = OracleTopo(geo, "D3Q19", "x")
    sr = np.sort(10.0 ** rng.uniform(-14, -4, rows))
    table = np.stack([sr, 0.02 + 0.15 * (1.0 + sr / 1e-9) ** -0.2], 1)
    f0 = oracle.rest_state(1, T.n_nodes, T.bulk, np.ones(T.n_nodes))
    f0[T.bulk] *= 1.0 + 1e-3 * rng.standard_normal((T.bulk.size, 19))
    force = np.array([1e-4, 2e-5, 0.0])
    fo, ro, vo, wo = oracle.run_rheology(1, T.neighbors, T.node_types, T.bulk, f0, table, force, 20)
    ctx = lbamd.Context(lbamd.D3Q19, precision)
    ctx.set_topology_grid(T.neighbors, T.node_types, T.bulk, T.positions)
    ctx.set_viscosity_table(table[:, 0], table[:, 1])
    ctx.upload_f(f0)
    ctx.step_rheology(20, force)
    v, w, b = ctx.download_vel(), ctx.download_scalar(lbamd.VISC), T.bulk
    f = ctx.download_f(1)[:, 0]
    ctx.close()
    if precision == lbamd.FP64:
        assert np.array_equal(v[b], vo[b]) and np.array_equal(w[b], wo[b]) and np.array_equal(f[b], fo[b])
    else:
        assert np.abs(v[b] - vo[b]).max() <= 1e-4 * np.abs(vo[b]).max()
