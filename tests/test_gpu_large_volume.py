"""Forward projection of volumes past 32-bit byte offsets (FP32: over 2^30 voxels) and close to
2^31 voxels (BF16): the array's last eight y rows hold values, and the projection is that of a
volume of these rows alone.  Both sides are FP32 sums of the same footprints, 1e-5 relative L2 (BF16
results rounded once more: 2^-8)."""

import numpy as np
import pytest

from bf16 import round_bits
from conftest import rel_l2

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu

ROWS = 8


def _geometry(n, ny, dnv):
    cfg = G.helical_config(sid=541, sdd=949, DNU=48, DNV=dnv, col_width=1.0239, col_height=1.0,
                           views_per_turn=6, turns=1, feed_mm_per_turn=0.0, N_xy=n, N_z=n,
                           voxel_xy=0.4, voxel_z=0.4)
    cfg["acq"]["first_view_angle"] = 10.0
    g = G.dd3_geometry(cfg)
    g.YN = ny
    g.imgYCenter = np.float32(-0.5 * ny * g.dx)  # the last row ends at the axis
    return g


@pytest.mark.parametrize("dnv", [16, 64])
@pytest.mark.parametrize("storage,n", [("f32", 1026), ("bf16", 1290)])
def test_last_rows_of_a_large_volume(storage, n, dnv, gpu_plan_factory):
    from ctrecon_amd._lib import check, lib
    from ctrecon_amd.plan import DeviceArray

    print(f"[large volume] {storage} {n}^3 rows={dnv}", flush=True)
    big, small = _geometry(n, n, dnv), _geometry(n, ROWS, dnv)
    assert n ** 3 > 2 ** 30 and n ** 3 < 2 ** 31
    v = np.random.default_rng(n).uniform(0, 1, small.vol_shape).astype(np.float32)
    if storage == "bf16":
        v = round_bits(v)
    dt = v.dtype
    d_small, d_big = DeviceArray.from_host(v), DeviceArray(big.vol_shape, dt)
    d_big.zero()
    check(lib().ctr_memcpy_h2d(d_big.ptr + d_big.nbytes - v.nbytes, v.ctypes.data, v.nbytes))
    out = []
    for g, d in ((big, d_big), (small, d_small)):
        plan, y = gpu_plan_factory(g), DeviceArray(g.prj_shape, dt)
        (plan.fp if storage == "f32" else plan.fp_bf16)(d, y)
        out.append(y.get())
        plan.close()
    d_big.free()
    if storage == "bf16":
        out = [(o.astype(np.uint32) << 16).view(np.float32) for o in out]
    assert np.all(np.any(out[1] != 0, axis=(1, 2)))
    err = rel_l2(out[0], out[1])
    print(f"  rel-L2 {err:.3e}", flush=True)
    assert err <= (1e-5 if storage == "f32" else 2.0 ** -8)
