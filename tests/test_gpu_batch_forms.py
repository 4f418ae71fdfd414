"""Batches whose scans run different back projectors: every scan's iterate has the bits of a batch
of its own with the same launch shapes, whatever the other scans need."""

import numpy as np
import pytest

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu

SUBSETS = 4


def _scan(dnv, nxy=20, nz=24, views=22, seed=0):
    cfg = G.helical_config(sid=200, sdd=380, DNU=48, DNV=dnv, col_width=1.3, col_height=40.0 / dnv,
                           views_per_turn=views, turns=1, feed_mm_per_turn=12.0, N_xy=nxy, N_z=nz,
                           voxel_xy=1.0, voxel_z=1.0)
    g = G.dd3_geometry(cfg, mask=G.fov_mask(nxy))
    b = np.random.default_rng(dnv + seed).uniform(0, 10, g.prj_shape).astype(np.float32)
    return g, b


def _run(scans, tuning, storage="f32", sweeps=2):
    """Iterates of a batch of the scans, and the plans' own buffers kept alive."""
    from ctrecon_amd.batch import Batch
    from ctrecon_amd.plan import DeviceArray, Plan

    plans = [Plan(g, 0) for g, _ in scans]
    for p in plans:
        p.set_storage(storage)
    bs = [DeviceArray.from_host(b) for _, b in scans]
    xs = [DeviceArray(g.vol_shape) for g, _ in scans]
    B = Batch(plans, xs, bs, SUBSETS)
    B.set_tuning(*tuning)
    for x in xs:
        x.zero()
    res, _ = B.sweeps(sweeps)
    out = [x.get() for x in xs]
    B.close()
    return out, res


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("grid", [0, 64])
def test_scans_over_256_rows_leave_the_others(grid, storage, gpu_plan_factory):
    print(f"[batch with 300 rows] grid={grid} storage={storage}", flush=True)
    scans = [_scan(64), _scan(300), _scan(16), _scan(100)]
    tuning = (False, grid, 5, grid)
    got, res = _run(scans, tuning, storage)
    for i, s in enumerate(scans):
        own, own_res = _run([s], tuning, storage)
        assert np.array_equal(got[i], own[0]), (i, s[0].DNV)
        assert np.allclose(res[:, i], own_res[:, 0], rtol=1e-12, atol=0)


def test_tuning_of_earlier_kernels_is_not_used(tmp_path, monkeypatch, gpu_plan_factory):
    """A stored line is found again by the same kernels, and not without their revision."""
    from ctrecon_amd.batch import Batch
    from ctrecon_amd.plan import DeviceArray, Plan

    print("[tuning revision]", flush=True)
    cache = tmp_path / "tuning.txt"
    monkeypatch.setenv("CTRECON_TUNE_CACHE", str(cache))
    g, b = _scan(40)
    p, db, x = Plan(g, 0), DeviceArray.from_host(b), DeviceArray(g.vol_shape)
    x.zero()

    def info():
        B = Batch([p], [x], [db], SUBSETS)
        i = B.info()
        B.close()
        return i

    assert info()["from_cache"] == 0
    line = cache.read_text().splitlines()[-1]
    assert info()["from_cache"] == 1
    # the line's key starts at the device's name without a revision
    key, values = line.split("\t")
    cache.write_text(key[key.index("gfx"):] + "\t" + values + "\n")
    assert info()["from_cache"] == 0


@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_tall_columns_in_z_groups(storage, gpu_plan_factory):
    """Columns over 2048 voxels: every number of z groups per lane adds a voxel's views in the same
    order as the scan's own solver (equal bits), beside a scan of short columns."""
    from ctrecon_amd.batch import Batch
    from ctrecon_amd.plan import DeviceArray, Plan

    print(f"[batch, tall columns] {storage}", flush=True)
    scans = [_scan(64, nxy=4, nz=2100), _scan(64), _scan(64, nxy=3, nz=2309, views=17)]
    ref = []
    for g, b in scans:
        p, x = Plan(g, 0), DeviceArray(g.vol_shape)
        p.set_storage(storage)
        x.zero()
        p.os_sart(x, DeviceArray.from_host(b), SUBSETS, 2)
        ref.append(x.get())
    plans = [Plan(g, 0) for g, _ in scans]
    for p in plans:
        p.set_storage(storage)
    bs = [DeviceArray.from_host(b) for _, b in scans]
    xs = [DeviceArray(g.vol_shape) for g, _ in scans]
    B = Batch(plans, xs, bs, SUBSETS)
    for zg in (0, 1, 2, 3, 4, 5):
        for grid, strided in ((0, False), (64, False), (64, True)):
            B.set_tuning(True, grid, zg, grid, strided, strided)
            for x in xs:
                x.zero()
            B.sweeps(2)
            for i, x in enumerate(xs):
                assert np.array_equal(x.get(), ref[i]), (zg, grid, strided, i)
    B.close()
