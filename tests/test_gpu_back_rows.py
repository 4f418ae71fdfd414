"""The windowed back projectors with staged rows against the FP64 oracle: detectors whose
rows fill one, two and four chunks of 64 and more than four (the unstaged form), one to five
columns per voxel (five: the general form), windows of one and of several 64-voxel passes,
shadows of two, three and more rows, unevenly spaced rows (the matched adjoint's other
kernel); and the set-up sums of OS-SART, which have to match the projections of ones down to
shadows that graze a voxel by a rounding error.

Bars: FP32 1e-5 relative L2, as the other parity tests (BF16 sinograms: the oracle on the
rounded values, FP32 sums, the same bar)."""

import numpy as np
import pytest

from bf16 import quantize
from conftest import rel_l2

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu


def _geometry(dnv, nz=33, vox=1.0, col=1.1, row=1.3, nxy=13, uneven=False, mask=True):
    cfg = G.helical_config(sid=200, sdd=380, DNU=19, DNV=dnv, col_width=col, col_height=row,
                           views_per_turn=35, turns=2, feed_mm_per_turn=9.0, N_xy=nxy, N_z=nz,
                           voxel_xy=vox, voxel_z=vox)
    g = G.dd3_geometry(cfg, mask=G.fov_mask(nxy) if mask else None)
    if uneven:
        g.zds = (g.zds + 0.2 * row * np.sin(np.arange(dnv))).astype(np.float32)
    return g


CASES = [dict(dnv=n) for n in (1, 2, 3, 8, 15, 16, 17, 32, 33, 40, 63, 64, 65, 100, 128, 129,
                               200, 256, 257)]
CASES += [
    dict(dnv=64, nz=200),                      # several passes
    dict(dnv=128, nz=331, vox=0.5),
    dict(dnv=16, nz=130, vox=0.25),
    dict(dnv=64, col=0.3),                     # many columns per voxel: the general form
    dict(dnv=16, col=0.3), dict(dnv=64, col=0.6), dict(dnv=64, col=3.0),
    dict(dnv=64, row=0.35),                    # more than three rows per voxel
    dict(dnv=16, row=0.35), dict(dnv=64, row=4.0),
    dict(dnv=64, nz=1), dict(dnv=40, nz=65, mask=False, nxy=7),
    dict(dnv=40, uneven=True), dict(dnv=12, uneven=True), dict(dnv=90, uneven=True),
]


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("kind", ["ref", "matched"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_back_rows(case, kind, storage, oracle, gpu_plan_factory):
    print(f"[back rows] {case} {kind} {storage}", flush=True)
    g = _geometry(**case)
    y = np.random.default_rng(2).uniform(-0.2, 1, g.prj_shape).astype(np.float32)
    plan = gpu_plan_factory(g)
    if storage == "bf16":
        y = quantize(y)
        got = plan.back_bf16(y, kind=kind)
    else:
        got = plan.back(y, kind=kind)
    ref = oracle.bp(g, y, "direct" if kind == "ref" else "adjoint")
    assert np.any(ref != 0)
    err = rel_l2(got, ref)
    print(f"  rel-L2 {err:.3e}", flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("dnv", [12, 40, 64, 80])
def test_set_up_sums_match_the_projections(dnv, gpu_plan_factory):
    """One OS-SART subset step from x = 0 on b = A 1: the residual over the row sums is 1 on
    every ray that meets the volume and 0 on the others, so the update is the back projection
    of that indicator over the back projection of ones -- for rays and voxels that are only
    grazed too, since each sum repeats the projection's own weights.  Bar: each ratio carries
    some FP32 roundings (2^-21), thousands of terms: 1e-4."""
    from ctrecon_amd.plan import DeviceArray

    print(f"[set-up sums] {dnv} rows", flush=True)
    g = _geometry(dnv, nz=61, nxy=25)
    plan = gpu_plan_factory(g)
    b = plan.forward(np.ones(g.vol_shape, np.float32))
    x = DeviceArray(g.vol_shape)
    x.zero()
    plan.os_sart(x, DeviceArray.from_host(b), 1, 1)
    x = x.get()
    num, den = (plan.back(y.astype(np.float32)) for y in (b != 0, np.ones_like(b)))
    seen = den != 0
    off = np.abs(x[seen] - num[seen] / den[seen])
    print(f"  seen {np.sum(seen)} of {x.size}, worst {off.max():.2e}", flush=True)
    assert np.any(seen) and np.all(x[~seen] == 0)
    assert off.max() <= 1e-4
