"""An infinity or NaN in one input cell reaches the outputs that the cell has a weight in, and
no others: the projectors' straight-line classes may read cells beside a footprint with weight
zero, and a wave that meets a value that is not finite runs its footprints' own cells only.

The weights are the FP64 oracle's projection of the cell's indicator; outputs of weight zero have
to be finite and keep the parity bar (1e-5 relative L2), those of a weight of more than 1e-4 of
the largest must not be finite (smaller ones may round to zero)."""

import numpy as np
import pytest

from conftest import rel_l2

from ctrecon_amd import geometry as G

pytestmark = pytest.mark.gpu

SCANS = [dict(dnv=16), dict(dnv=40), dict(dnv=64, nz=90), dict(dnv=80), dict(dnv=64, row=3.5),
         dict(dnv=16, col=0.4)]


def _geometry(dnv, nz=33, row=1.3, col=1.1):
    cfg = G.helical_config(sid=200, sdd=380, DNU=25, DNV=dnv, col_width=col, col_height=row,
                           views_per_turn=35, turns=2, feed_mm_per_turn=9.0, N_xy=13, N_z=nz,
                           voxel_xy=1.0, voxel_z=1.0)
    return G.dd3_geometry(cfg, mask=G.fov_mask(13))


def _check(got, ref, w):
    bad = ~np.isfinite(got)
    print(f"  {bad.sum()} not finite of {bad.size}, {np.sum(w > 0)} with a weight", flush=True)
    assert np.all(bad[w > 1e-4 * w.max()]) and not np.any(bad[w == 0])
    assert rel_l2(got[w == 0], ref[w == 0]) <= 1e-5


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("scan", SCANS, ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_forward(scan, value, oracle, gpu_plan_factory):
    print(f"[not finite] forward {scan} {value}", flush=True)
    g = _geometry(**scan)
    vol = np.random.default_rng(1).uniform(0, 1, g.vol_shape).astype(np.float32)
    one = np.zeros_like(vol)
    at = (7, 5, g.ZN // 2)
    one[at] = 1
    clean, vol[at] = oracle.fp(g, vol, "direct"), value
    _check(gpu_plan_factory(g).forward(vol), clean, oracle.fp(g, one, "direct"))


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("kind", ["ref", "matched"])
@pytest.mark.parametrize("scan", SCANS, ids=lambda c: ",".join(f"{k}={v}" for k, v in c.items()))
def test_back(scan, kind, value, oracle, gpu_plan_factory):
    print(f"[not finite] back {kind} {scan} {value}", flush=True)
    g = _geometry(**scan)
    y = np.random.default_rng(2).uniform(0, 1, g.prj_shape).astype(np.float32)
    one = np.zeros_like(y)
    at = (g.PN // 2, 12, g.DNV // 2)
    one[at] = 1
    model = "direct" if kind == "ref" else "adjoint"
    clean, y[at] = oracle.bp(g, y, model), value
    _check(gpu_plan_factory(g).back(y, kind=kind), clean, np.abs(oracle.bp(g, one, model)))
