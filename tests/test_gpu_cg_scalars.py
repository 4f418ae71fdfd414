"""CG with its scalars on the device: the residuals of a long call, which are read back in
groups of 32, are those of shorter calls from the same start (equal bits), and the iterate is the
FP64 oracle's to the bar of the other CG tests."""

import numpy as np
import pytest

from conftest import rel_l2

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def test_residuals_of_long_calls(oracle, gpu_plan_factory):
    from ctrecon_amd.plan import DeviceArray

    print("[CG scalars]", flush=True)
    cfg = G.helical_config(sid=200, sdd=380, DNU=23, DNV=8, col_width=1.1, col_height=1.3,
                           views_per_turn=24, turns=2, feed_mm_per_turn=6.0, N_xy=9, N_z=10,
                           voxel_xy=1.0, voxel_z=1.0)
    g = G.dd3_geometry(cfg, mask=G.fov_mask(9))
    vol = np.random.default_rng(1).uniform(0, 1, g.vol_shape).astype(np.float32)
    plan = gpu_plan_factory(g)
    b = plan.forward(vol)
    db = DeviceArray.from_host(b)

    def run(n):
        x = DeviceArray(g.vol_shape)
        x.zero()
        return np.asarray(plan.conjgrad(x, db, n, "matched")), x.get()

    full, _ = run(70)
    assert full.size == 70 and np.all(np.isfinite(full))
    for n in (1, 2, 31, 32, 33, 64, 65):
        assert np.array_equal(run(n)[0], full[:n]), n
    res, x = run(3)
    xr, rr = oracle.conjgrad(g, b, iterNum=3, bp_kind="matched")
    assert rel_l2(x, xr) <= 1e-4 and np.allclose(res, rr, rtol=1e-4)
