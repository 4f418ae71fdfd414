"""Residuals of the integral-image method.  Its forward projector writes one pair of partial sums
per 256 rays, the direct method's one per workgroup of lane groups: more, where a detector's rows
do not fill the groups.  The partial sums' buffers are first filled by the direct method; the
residuals after a change to the integral images are then the FP64 oracle's, to 1e-5 for one
projection (the method's bar) and to 1e-4 for sweeps (the bar of the solver's iterates)."""

import numpy as np
import pytest

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def _scan(dnv):
    cfg = G.helical_config(sid=200, sdd=380, DNU=40, DNV=dnv, col_width=1.2, col_height=16.0 / dnv,
                           views_per_turn=20, turns=2, feed_mm_per_turn=6.0, N_xy=16, N_z=12,
                           voxel_xy=1.0, voxel_z=1.0)
    return G.dd3_geometry(cfg, mask=G.fov_mask(16))


@pytest.mark.parametrize("dnv", [12, 24, 40])
def test_sat_residuals_after_the_direct_method(dnv, oracle, gpu_plan_factory):
    from ctrecon_amd.plan import DeviceArray, Sart

    print(f"[SAT residuals] rows={dnv}", flush=True)
    g = _scan(dnv)
    rng = np.random.default_rng(dnv)
    x0 = rng.uniform(0, 1, g.vol_shape).astype(np.float32)
    b = rng.uniform(0, 20, g.prj_shape).astype(np.float32)
    plan = gpu_plan_factory(g)
    dx, db = DeviceArray.from_host(x0), DeviceArray.from_host(b)
    d = b - oracle.fp(g, x0, "sat")
    ref = np.linalg.norm(d) / np.linalg.norm(b)
    got = []
    for method in ("direct", "sat"):
        plan.set_method(method)
        got.append(plan.residual(dx, db))
    print(f"  residual {got} oracle {ref}", flush=True)
    assert np.allclose(got, ref, rtol=1e-5)
    plan.set_method("direct")
    s = Sart(plan, db, 4)
    s.set_graph(False)
    s.sweeps(dx, 1)
    plan.set_method("sat")
    dx.zero()
    res, _, _ = s.sweeps(dx, 2)
    s.close()
    _, rr = oracle.os_sart(g, b, osNum=4, iterNum=2, bp_kind="ref")
    print(f"  sweeps {res} oracle {rr}", flush=True)
    assert np.allclose(res, rr, rtol=1e-4)


def test_sat_solver_residuals(oracle, gpu_plan_factory):
    """os_sart as a call of its own, with the stopping rule on its residual."""
    from ctrecon_amd.plan import DeviceArray

    print("[SAT os_sart residuals]", flush=True)
    g = _scan(24)
    b = np.random.default_rng(2).uniform(0, 20, g.prj_shape).astype(np.float32)
    plan = gpu_plan_factory(g)
    plan.set_method("sat")
    _, rr = oracle.os_sart(g, b, osNum=4, iterNum=3, bp_kind="ref")
    assert rr[1] < rr[0]
    dx = DeviceArray(g.vol_shape)
    dx.zero()
    res, _, _ = plan.os_sart_run(dx, DeviceArray.from_host(b), 4, 3, "ref",
                                 stop_resid=float(0.5 * (rr[0] + rr[1])))
    assert len(res) == 2 and np.allclose(res, rr[:2], rtol=1e-4)
