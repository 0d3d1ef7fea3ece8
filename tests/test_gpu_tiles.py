"""Small D2Q9 lists advance several steps per launch in long calls
(csrc/tile2d.hpp): one long call and calls of some launches against calls of 5
steps, which are too short for that, bit for bit,
FP64 and FP32S, BGK and TRT.  Boxes narrower than a tile's halo along the
periodic axis, smaller than a tile, one cell short of and beyond tiles, closed
along x, and random solids."""
import numpy as np
import pytest

import lbamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [lbamd.FP64, lbamd.FP32S])
@pytest.mark.parametrize("shape,periodic,solids,op", [
    ((2, 9), "x", 0.0, "bgk"), ((5, 14), "x", 0.2, "trt"), ((12, 14), "x", 0.3, "bgk"),
    ((13, 27), "x", 0.3, "bgk"), ((35, 26), "x", 0.3, "trt"), ((24, 50), "", 0.25, "bgk"),
    ((61, 39), "x", 0.4, "bgk")])
def test_long_call_equals_short_calls(gpu_available, precision, shape, periodic, solids, op):
    rng = np.random.default_rng(shape[0])
    geo = (rng.random(shape) >= solids).astype(np.int32)
    geo[:, 0] = geo[:, -1] = 0
    if "x" not in periodic:
        geo[0] = geo[-1] = 0
    topo = lbamd.Topology.from_geometry(geo, lbamd.D2Q9, periodic)
    w = np.array([4.0, 1.0] * 4 + [16.0]) / 36.0
    f0 = w * (1.0 + 1e-3 * rng.standard_normal((topo.n_nodes, 9)))
    out = []
    for chunks in ([260], [100, 8, 152], [5] * 52):
        ctx = lbamd.Context(lbamd.D2Q9, precision)
        ctx.set_topology_from(topo)
        assert ctx.layout == 2, ctx.layout_note
        ctx.upload_f(f0)
        for n in chunks:
            if op == "trt":
                ctx.step_trt(n, 1.0, 0.875, (1e-5, 2e-6))
            else:
                ctx.step_bgk(n, 0.9, (1e-5, 2e-6))
        b = topo.bulk()
        out.append((ctx.download_f(1)[b], ctx.download_scalar(lbamd.RHO)[b], ctx.download_vel()[b]))
        ctx.close()
    for plain, a, b in zip(out[2], *out[:2]):
        assert np.isfinite(plain).all() and np.array_equal(a, plain) and np.array_equal(b, plain)
