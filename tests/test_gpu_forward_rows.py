"""The forward projector's work mappings against the FP64 oracle: detectors whose rows fill,
underfill and overfill a wave (groups of 8, 16 and 32 rows, one column per wave, several
items per column), and the classes of a slice -- one to five in-plane cells, two or three z
taps, z runs over 64 and over 128 cells, more than two cells of height, footprints past both
ends of the volume, the array's last column.

Bars: FP32 1e-5 relative L2, as the other parity tests; BF16 (the oracle on the rounded
volume, FP32 sums, one rounding of each result by at most 2^-9) 2^-9."""

import numpy as np
import pytest

from bf16 import quantize
from conftest import rel_l2

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def _geometry(dnv, nz=21, vox=1.0, col=1.1, row=1.3, nxy=27, turns=2, feed=None, mask=True):
    cfg = G.helical_config(sid=200, sdd=380, DNU=23, DNV=dnv, col_width=col, col_height=row,
                           views_per_turn=11, turns=turns,
                           feed_mm_per_turn=12.0 if feed is None else feed, N_xy=nxy, N_z=nz,
                           voxel_xy=vox, voxel_z=vox)
    return G.dd3_geometry(cfg, mask=G.fov_mask(nxy) if mask else None)


CASES = [dict(dnv=n) for n in (1, 2, 7, 8, 9, 12, 16, 17, 24, 31, 32, 33, 40, 63, 64, 65, 80,
                               128, 130)]
CASES += [
    dict(dnv=64, nz=150, feed=0.0),                      # wholly inside: three taps, one run
    dict(dnv=64, nz=200, feed=0.0, row=1.9),             # runs over 64 cells
    dict(dnv=64, nz=301, feed=0.0, row=3.7),             # runs over 64, heights near 2
    dict(dnv=64, nz=331, feed=0.0, row=4.9),             # heights over 2: the general form
    dict(dnv=64, nz=150, feed=0.0, row=0.6, col=0.4),    # two taps, one or two cells
    dict(dnv=64, nz=99, col=4.1, feed=0.0),              # three or four cells
    dict(dnv=64, nz=99, col=9.0, feed=0.0),              # five and more: the general form
    dict(dnv=16, nz=99, col=4.1, feed=0.0),
    dict(dnv=16, nz=99, col=9.0, feed=0.0),
    dict(dnv=16, nz=44, row=4.9),
    dict(dnv=64, nz=40, mask=False, col=2.0),            # the array's last column is read
    dict(dnv=16, nz=40, mask=False, col=2.0),
    dict(dnv=64, nz=1), dict(dnv=64, nz=3, nxy=1, mask=False), dict(dnv=8, nz=1, nxy=2, mask=False),
]


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_forward_rows(case, storage, oracle, gpu_plan_factory):
    print(f"[forward rows] {case} {storage}", flush=True)
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
