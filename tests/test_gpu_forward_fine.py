"""The forward projector's form for fine voxels and wide columns against the FP64 oracle: one to
thirteen cells of a slice, rows up to twelve cells high, both ends of the volume, the array's last
column, volumes of few voxels.  Bars: FP32 1e-5 relative L2, BF16 2^-9 (one rounding of each
result), as the other forms.  A batch in which one scan needs this form leaves the other scans'
bits as they are."""

import numpy as np
import pytest

from bf16 import quantize
from conftest import rel_l2
from test_gpu_batch_forms import _run, _scan

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def _geometry(dnv, nxy=21, nz=23, vox=1.0, vz=None, col=1.1, row=1.3, feed=3.0, mask=True):
    cfg = G.helical_config(sid=200, sdd=380, DNU=19, DNV=dnv, col_width=col, col_height=row,
                           views_per_turn=13, turns=2, feed_mm_per_turn=feed, N_xy=nxy, N_z=nz,
                           voxel_xy=vox, voxel_z=vox if vz is None else vz)
    return G.dd3_geometry(cfg, mask=G.fov_mask(nxy) if mask else None)


CASES = [dict(dnv=n, **k) for n in (1, 5, 8, 16, 33, 64, 70, 257)
         for k in (dict(vox=0.15), dict(vz=0.15, nz=61), dict(col=6.0, mask=False))]
CASES += [
    dict(dnv=64, vox=0.06, feed=0.5), dict(dnv=16, vox=0.06, feed=0.5),   # 13 cells, 12 high
    dict(dnv=64, vz=0.33, nz=400, feed=0.0), dict(dnv=16, vz=0.33, nz=150, feed=0.0),
    dict(dnv=64, vz=0.31, row=1.2, mask=False), dict(dnv=16, vz=0.31, row=1.2, mask=False),
    dict(dnv=64, col=14.0, row=4.5, nz=40), dict(dnv=8, col=14.0, row=4.5, nz=40),
    dict(dnv=64, nxy=2, nz=1, vox=0.2, mask=False), dict(dnv=8, nxy=1, nz=4, vox=0.2, mask=False),
    dict(dnv=8, nxy=1, nz=3, vox=0.2, mask=False),
]


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_forward_fine(case, storage, oracle, gpu_plan_factory):
    print(f"[forward fine] {case} {storage}", flush=True)
    g = _geometry(**case)
    vol = np.random.default_rng(1).uniform(0, 1, g.vol_shape).astype(np.float32)
    plan = gpu_plan_factory(g)
    if storage == "bf16":
        vol = quantize(vol)
        got, bar = plan.forward_bf16(vol), 2.0 ** -9
    else:
        got, bar = plan.forward(vol), 1e-5
    ref = oracle.fp(g, vol, "direct")
    assert np.any(ref != 0)
    err = rel_l2(got, ref)
    print(f"  rel-L2 {err:.3e}", flush=True)
    assert err <= bar
    assert np.all(got[ref == 0] == 0)


@pytest.mark.parametrize("case", [dict(dnv=64, vox=0.15), dict(dnv=16, vz=0.15, nz=61),
                                  dict(dnv=16, col=6.0)],
                         ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_fine_solver(case, oracle, gpu_plan_factory):
    """Row sums and residuals of the form, through the solver (its iterates' bar, 1e-4)."""
    from ctrecon_amd.plan import DeviceArray

    print(f"[fine solver] {case}", flush=True)
    g = _geometry(**case)
    vol = np.random.default_rng(3).uniform(0, 1, g.vol_shape).astype(np.float32)
    b = oracle.fp(g, vol, "direct").astype(np.float32)
    x = DeviceArray(g.vol_shape)
    x.zero()
    res = gpu_plan_factory(g).os_sart(x, DeviceArray.from_host(b), 3, 2, "ref")
    xr, rr = oracle.os_sart(g, b, osNum=3, iterNum=2, bp_kind="ref")
    assert rel_l2(x.get(), xr) <= 1e-4 and np.allclose(res, rr, rtol=1e-4)


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("case", [dict(dnv=64, vz=0.15, nz=61), dict(dnv=16, vz=0.15, nz=61),
                                  dict(dnv=64, col=6.0), dict(dnv=16, col=6.0)],
                         ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_fine_not_finite(case, value, oracle, gpu_plan_factory):
    print(f"[fine, not finite] {case} {value}", flush=True)
    g = _geometry(**case)
    vol = np.random.default_rng(1).uniform(0, 1, g.vol_shape).astype(np.float32)
    one = np.zeros_like(vol)
    at = (10, 9, g.ZN // 2)
    one[at] = 1
    clean, w = oracle.fp(g, vol, "direct"), oracle.fp(g, one, "direct")
    vol[at] = value
    got = gpu_plan_factory(g).forward(vol)
    bad = ~np.isfinite(got)
    assert np.all(bad[w > 1e-4 * w.max()]) and not np.any(bad[w == 0])
    assert rel_l2(got[w == 0], clean[w == 0]) <= 1e-5


@pytest.mark.parametrize("grid", [0, 64])
@pytest.mark.parametrize("colw", [False, True])
def test_batch_with_a_fine_scan(colw, grid, gpu_plan_factory):
    print(f"[batch with a fine scan] colw={colw} grid={grid}", flush=True)
    fine = _geometry(64, vox=0.15)
    b = np.random.default_rng(4).uniform(0, 10, fine.prj_shape).astype(np.float32)
    scans = [_scan(64), (fine, b), _scan(64, nxy=17, nz=31) if colw else _scan(16)]
    tuning = (colw, grid, 5, grid)
    got, _ = _run(scans, tuning)
    for i, s in enumerate(scans):
        assert np.array_equal(got[i], _run([s], tuning)[0][0]), i
