"""A plan's tables, which one launch computes for all (view, column) pairs, mask cells, slices
and rows, against the FP64 oracle: sizes around a workgroup of pairs and of cells, one view,
one column, grids of unequal sides, a mask with empty slices, uneven rows, an off-centre
volume.  Bar: 1e-5 relative L2, as the other parity tests; also the host-buffer call gives the
plan's bits, which runs without the wait that ends a plan's creation."""

import dataclasses

import numpy as np
import pytest

from conftest import rel_l2

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def _geometry(dnu, dnv, views, nx, ny, nz, uneven):
    cfg = G.helical_config(sid=200, sdd=380, DNU=dnu, DNV=dnv, col_width=60.0 / max(dnu, 2),
                           col_height=1.3, views_per_turn=views, turns=1, feed_mm_per_turn=9.0,
                           N_xy=max(nx, ny), N_z=nz, voxel_xy=1.0, voxel_z=1.0)
    g = G.dd3_geometry(cfg)
    rng = np.random.default_rng(views)
    mask = np.ones((ny, nx), np.uint8)
    if min(nx, ny) > 4:
        mask[:2] = 0
        mask[:, -1] = 0
        mask[ny // 2] = 0
    zds = np.sort(g.zds + rng.uniform(-0.3, 0.3, dnv)).astype(np.float32) if uneven else g.zds
    return dataclasses.replace(g, XN=nx, YN=ny, mask=mask.ravel(), imgXCenter=1.7,
                               imgYCenter=-2.3, zds=zds)


@pytest.mark.parametrize("dnu,dnv,views,nx,ny,nz,uneven", [
    (1, 1, 1, 1, 1, 1, False), (1, 3, 2, 3, 7, 5, True), (15, 5, 16, 16, 16, 9, False),
    (16, 8, 15, 17, 15, 9, True), (31, 4, 8, 13, 29, 12, False), (254, 2, 3, 33, 8, 6, True),
    (37, 260, 7, 9, 31, 40, True),
])
def test_tables(dnu, dnv, views, nx, ny, nz, uneven, oracle, gpu_plan_factory):
    from ctrecon_amd import dd3 as D
    from ctrecon_amd._lib import check, lib

    print(f"[plan tables] {dnu}x{dnv} detector, {views} views, {nx}x{ny}x{nz}", flush=True)
    g = _geometry(dnu, dnv, views, nx, ny, nz, uneven)
    vol = np.random.default_rng(2).uniform(0, 1, g.vol_shape).astype(np.float32)
    got = gpu_plan_factory(g).forward(vol)
    ref = oracle.fp(g, vol, "direct")
    assert rel_l2(got, ref) <= 1e-5 if np.any(ref) else not np.any(got)
    argv, keep = D._geo_argv(g)
    prj = np.empty(got.size, np.float32)
    flat = np.ascontiguousarray(vol.ravel())
    check(lib().ctr_dd3_proj(*argv, flat.ctypes.data, prj.ctypes.data, g.dx, g.dz,
                             g.mask.ctypes.data, 0, 0))
    assert np.array_equal(prj, got.ravel())
