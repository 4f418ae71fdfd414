"""The windowed back projectors with several views per wave, for detectors of few rows, against
the FP64 oracle: two to eight groups of lanes with and without idle lanes, windows that fill a
group, overflow it (a second pass) or reach past the volume, fewer views than groups, columns
whose sums fill the groups' share of LDS and columns past it (one view at a time); and a batch
of scans that take both forms, which has to give the bits of each scan by itself.

Bars: FP32 1e-5 relative L2, as the other parity tests."""

import numpy as np
import pytest

from conftest import rel_l2

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def _geometry(dnv, nz=33, vox=1.0, row=1.3, nxy=13, views=35, turns=2, col=1.1):
    cfg = G.helical_config(sid=200, sdd=380, DNU=19, DNV=dnv, col_width=col, col_height=row,
                           views_per_turn=views, turns=turns, feed_mm_per_turn=9.0, N_xy=nxy,
                           N_z=nz, voxel_xy=vox, voxel_z=vox)
    return G.dd3_geometry(cfg, mask=G.fov_mask(nxy))


CASES = [dict(dnv=n) for n in (4, 5, 6, 7, 9, 10, 11, 12, 13, 18, 20, 21, 22, 24, 30, 31)]
CASES += [
    dict(dnv=16, vox=0.43),                  # windows of 25 of 32 lanes
    dict(dnv=16, vox=0.33),                  # windows of more than 32 voxels on the far side
    dict(dnv=32, vox=0.7, nxy=41),           # both passes
    dict(dnv=16, vox=2.5),                   # fewer voxels than rows
    dict(dnv=16, views=1, turns=1), dict(dnv=16, views=2, turns=1), dict(dnv=8, views=7, turns=1),
    dict(dnv=16, views=130, turns=1),        # three blocks of 64 views
    dict(dnv=16, nz=1), dict(dnv=16, nz=2, nxy=3),
    dict(dnv=16, nz=512), dict(dnv=16, nz=520), dict(dnv=24, nz=768, vox=1.1),
    dict(dnv=16, nz=772),
    dict(dnv=16, col=4.0), dict(dnv=16, col=0.5), dict(dnv=20, row=3.5),
]


@pytest.mark.parametrize("kind", ["ref", "matched"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_back_packed(case, kind, oracle, gpu_plan_factory):
    print(f"[back packed] {case} {kind}", flush=True)
    g = _geometry(**case)
    y = np.random.default_rng(2).uniform(-0.2, 1, g.prj_shape).astype(np.float32)
    got = gpu_plan_factory(g).back(y, kind=kind)
    ref = oracle.bp(g, y, "direct" if kind == "ref" else "adjoint")
    assert np.any(ref != 0)
    err = rel_l2(got, ref)
    print(f"  rel-L2 {err:.3e}", flush=True)
    assert err <= 1e-5


def test_batch_of_both_forms(gpu_plan_factory):
    """(The forward projector's rows per wave are a batch's, not a scan's own: the bits to
    match are those of a batch of the one scan with the same tuning.)"""
    from ctrecon_amd.batch import Batch
    from ctrecon_amd.plan import DeviceArray

    print("[back packed] batch", flush=True)

    def sweeps(scans):
        xs = [DeviceArray(p.g.vol_shape) for p, _ in scans]
        for x in xs:
            x.zero()
        B = Batch([p for p, _ in scans], xs, [b for _, b in scans], 5)
        B.set_tuning(False, 0, 0, 0)
        B.sweeps(2)
        return [x.get() for x in xs]

    scans = []
    for dnv, nz in ((16, 33), (40, 29), (8, 70), (24, 12)):
        g = _geometry(dnv, nz)
        plan = gpu_plan_factory(g)
        vol = np.random.default_rng(dnv).uniform(0, 1, g.vol_shape).astype(np.float32)
        scans.append((plan, DeviceArray.from_host(plan.forward(vol))))
    for got, scan in zip(sweeps(scans), scans):
        assert np.any(got)
        assert np.array_equal(got, sweeps([scan])[0])
