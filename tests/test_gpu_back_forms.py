"""The back projectors' forms by the number of views and the size of the voxels: one and two views,
and coarse voxels, with rows staged view by view; several views per wave from 16 views on.  FP64
oracle: projections 1e-5, the solver's iterates 1e-4 (their bars elsewhere); BF16 sinograms are
exact inputs.  A batch runs each scan and subset step in the form of the scan's own solver (equal
bits)."""

import numpy as np
import pytest

from bf16 import quantize, round_bits
from conftest import rel_l2
from test_gpu_batch_forms import _run

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def _geometry(dnv, views=8, nxy=15, nz=26, vox=1.0, col=1.3, feed=6.0):
    cfg = G.helical_config(sid=200, sdd=380, DNU=41, DNV=dnv, col_width=col,
                           col_height=min(1.5, 60.0 / dnv), views_per_turn=views, turns=1,
                           feed_mm_per_turn=feed, N_xy=nxy, N_z=nz, voxel_xy=vox, voxel_z=vox)
    cfg["acq"]["first_view_angle"] = 20.0
    return G.dd3_geometry(cfg, mask=G.fov_mask(nxy))


GRIDS = [dict(), dict(vox=3.1, nxy=9, nz=11), dict(col=0.2), dict(vox=3.1, col=0.3, nxy=7, nz=9),
         dict(vox=8.0, nxy=5, nz=6)]


@pytest.mark.parametrize("kind", ["ref", "matched"])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()) or
                         "plain")
@pytest.mark.parametrize("dnv", [1, 16, 33, 64, 65, 128, 129, 256])
def test_view_counts(dnv, grid, kind, oracle, gpu_plan_factory):
    from ctrecon_amd.plan import DeviceArray

    print(f"[back forms] rows={dnv} {grid} {kind}", flush=True)
    g = _geometry(dnv, views=35, **grid)
    plan = gpu_plan_factory(g)
    y = quantize(np.random.default_rng(dnv).uniform(0, 1, g.prj_shape).astype(np.float32))
    out = DeviceArray(g.vol_shape)
    for first, step, n in ((0, 1, 1), (7, 1, 1), (3, 5, 2), (1, 2, 3), (4, 2, 15), (1, 2, 16)):
        views = first + step * np.arange(n)
        # the library reads the views' frames one after the other
        d_v = DeviceArray.from_host(np.ascontiguousarray(y[views]))
        plan.bp(d_v, out, first, step, n, kind=kind)
        ref = oracle.bp(g.subset(views), y[views], "direct" if kind == "ref" else "adjoint")
        err = rel_l2(out.get(), ref)
        print(f"  {n} views: rel-L2 {err:.3e}", flush=True)
        assert err <= 1e-5
        d_v = DeviceArray.from_host(np.ascontiguousarray(round_bits(y)[views]))
        plan.bp_bf16(d_v, out, first, step, n, kind=kind)
        assert rel_l2(out.get(), ref) <= 1e-5


@pytest.mark.parametrize("grid", [dict(), dict(vox=3.1, nxy=9, nz=11)], ids=["fine", "coarse"])
@pytest.mark.parametrize("dnv", [16, 64, 100, 200])
@pytest.mark.parametrize("subsets", [8, 5, 3])
def test_solver_of_few_views(dnv, subsets, grid, oracle, gpu_plan_factory):
    """Subsets of one, of one and two, and of two and three views: column sums, update, residual."""
    from ctrecon_amd.plan import DeviceArray

    print(f"[few views per subset] rows={dnv} subsets={subsets} {grid}", flush=True)
    g = _geometry(dnv, **grid)
    vol = np.random.default_rng(3).uniform(0, 1, g.vol_shape).astype(np.float32)
    b = oracle.fp(g, vol, "direct").astype(np.float32)
    x = DeviceArray(g.vol_shape)
    x.zero()
    res = gpu_plan_factory(g).os_sart(x, DeviceArray.from_host(b), subsets, 2, "ref")
    xr, rr = oracle.os_sart(g, b, osNum=subsets, iterNum=2, bp_kind="ref")
    assert rel_l2(x.get(), xr) <= 1e-4 and np.allclose(res, rr, rtol=1e-4)


@pytest.mark.parametrize("grid", [0, 64])
def test_batch_of_many_forms(grid, gpu_plan_factory):
    """Subset steps of two and three views, of fifteen and sixteen, coarse and fine scans."""
    print(f"[batch of many forms] grid={grid}", flush=True)
    scans = []
    for k, (dnv, views, more) in enumerate([(64, 9, {}), (16, 61, {}), (64, 11, dict(vox=3.1, nxy=9)),
                                            (130, 10, {}), (300, 9, {}), (16, 9, {}), (80, 6, {})]):
        g = _geometry(dnv, views=views, **more)
        scans.append((g, np.random.default_rng(k).uniform(0, 9, g.prj_shape).astype(np.float32)))
    tuning = (False, grid, 5, grid)
    got, res = _run(scans, tuning)
    for i, s in enumerate(scans):
        own, own_res = _run([s], tuning)
        assert np.array_equal(got[i], own[0]), (i, s[0].DNV, s[0].PN)
        assert np.allclose(res[:, i], own_res[:, 0], rtol=1e-12, atol=0)


def test_batch_has_the_solver_bits(gpu_plan_factory):
    """One column per wave (64 rows) in both: the batch's iterates are the solver's."""
    from ctrecon_amd.plan import DeviceArray, Plan

    print("[batch = solver over forms]", flush=True)
    scans = []
    for k, (views, more) in enumerate([(9, {}), (4, {}), (11, dict(vox=3.1, nxy=9)), (70, {})]):
        g = _geometry(64, views=views, **more)
        scans.append((g, np.random.default_rng(k).uniform(0, 9, g.prj_shape).astype(np.float32)))
    got, _ = _run(scans, (True, 0, 5, 0))
    for i, (g, b) in enumerate(scans):
        x = DeviceArray(g.vol_shape)
        x.zero()
        Plan(g, 0).os_sart(x, DeviceArray.from_host(b), 4, 2)
        assert np.array_equal(got[i], x.get()), i


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("dnv,grid", [(64, dict()), (64, dict(vox=3.1, nxy=9)), (64, dict(col=0.2)),
                                      (100, dict()), (200, dict())])
def test_not_finite(dnv, grid, value, oracle, gpu_plan_factory):
    print(f"[back forms, not finite] rows={dnv} {grid} {value}", flush=True)
    g = _geometry(dnv, views=2, **grid)
    y = np.random.default_rng(2).uniform(0, 1, g.prj_shape).astype(np.float32)
    one = np.zeros_like(y)
    at = (1, 20, g.DNV // 2)
    one[at] = 1
    clean, w = oracle.bp(g, y, "direct"), np.abs(oracle.bp(g, one, "direct"))
    y[at] = value
    got = gpu_plan_factory(g).back(y, kind="ref")
    bad = ~np.isfinite(got)
    assert np.any(w > 0) and np.all(bad[w > 1e-4 * w.max()]) and not np.any(bad[w == 0])
    assert rel_l2(got[w == 0], clean[w == 0]) <= 1e-5
