"""The network on grids that take the convolutions' large boxes, their runs along z, the
64-bit loads of very long (x, z) slices, and more boxes than a weight gradient has workgroups.

A voxel's value depends on the inputs within 2 + 2*2 + 2*4 + 2*2 + 2 = 20 voxels, and up to 4
more for the alignment of the coarser levels; and every configuration adds the same products
in the same order.  So a part of a large grid's output has the bits of the same part of a crop
that reaches 32 voxels further (or to the grid's edge), and a loss confined to that part has
the crop's gradient, up to the BF16 rounding of gradients that differ by the factor V / V_crop
(the bar of the other gradient tests, 3e-2).  The crops take the small boxes, which the other
tests compare with the oracle."""

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

SHAPES = [
    (68, 68, 128),  # boxes of 8 x 8 lines, ragged in y and x
    (36, 1028, 256),  # runs of four boxes along z
    (4, 2048, 3296),  # ten lines y of 16 channels span more than 2 GiB
]


def _part(n, where, keep, margin):
    """(start, stop) of the crop and of the part compared along an axis of n voxels."""
    if n < keep + margin:
        return (0, n), (0, n)
    if where == "low":
        return (0, keep + margin), (0, keep)
    if where == "high":
        return (n - keep - margin, n), (n - keep, n)
    if n < keep + 2 * margin:
        return (0, n), (0, n)
    s = (n // 2 - margin) // 4 * 4
    return (s, s + keep + 2 * margin), (s + margin, s + margin + keep)


@pytest.mark.parametrize("where", ["low", "mid", "high"])
@pytest.mark.parametrize("shape", SHAPES)
def test_part_of_a_large_grid(shape, where, gpu_plan_factory):
    from ctrecon_amd.plan import DeviceArray
    from ctrecon_amd.unet import LAYERS, UNet, init_params

    print(f"[unet boxes] grid={shape} {where}", flush=True)
    rng = np.random.default_rng(11)
    x = rng.random(shape, np.float32) * 2
    d = (rng.random(shape, np.float32) - 0.5) * 0.1
    p = init_params(12)
    p += np.random.default_rng(13).normal(0, 0.01, p.size).astype(np.float32)
    net = UNet(p, (1.0, 20.0, 1.0))

    def forward(a, b):
        out = DeviceArray(a.shape)
        net.forward(DeviceArray.from_host(a), DeviceArray.from_host(b), out)
        return out.get()

    axes = [_part(n, where, k, 32) for n, k in zip(shape, (8, 8, 32))]
    crop = tuple(slice(*c) for c, _ in axes)
    big = tuple(slice(*k) for _, k in axes)
    small = tuple(slice(k[0] - c[0], k[1] - c[0]) for c, k in axes)
    xc, dc = (np.ascontiguousarray(a[crop]) for a in (x, d))
    out, outc = forward(x, d), forward(xc, dc)
    assert np.isfinite(out).all()
    assert np.array_equal(out[big], outc[small])

    bump = rng.normal(0, 0.05, outc[small].shape).astype(np.float32)
    out[big] += bump
    outc[small] += bump
    _, g = net.loss_grad(*(DeviceArray.from_host(a) for a in (x, d, out)))
    _, gc = net.loss_grad(*(DeviceArray.from_host(a) for a in (xc, dc, outc)))
    gc *= outc.size / out.size
    o = 0
    errs = []
    for ci, co in LAYERS:
        for n in (27 * ci * co, co):
            errs.append(rel_l2(g[o:o + n], gc[o:o + n]))
            o += n
    errs.append(rel_l2(g[o:], gc[o:]))
    print(f"  worst gradient rel-L2 {max(errs):.2e}", flush=True)
    assert max(errs) <= 3e-2


def test_gradient_over_many_boxes(gpu_plan_factory):
    from bf16 import quantize
    from ctrecon_amd.plan import DeviceArray
    from ctrecon_amd.unet import LAYERS, UNet, init_params
    from oracle import unet_oracle as U

    shape, scales = (36, 68, 96), (1.0, 20.0, 0.05)
    print(f"[unet boxes] gradient, grid={shape}", flush=True)
    rng = np.random.default_rng(21)
    x = rng.uniform(0, 2, shape).astype(np.float32)
    d, t = (rng.normal(0, 0.05, shape).astype(np.float32) for _ in range(2))
    p = init_params(22)
    p += np.random.default_rng(23).normal(0, 0.01, p.size).astype(np.float32)
    loss, g = UNet(p, scales).loss_grad(*(DeviceArray.from_host(a) for a in (x, d, t)))
    q = lambda a: quantize(np.asarray(a, np.float32)).astype(np.float64)
    loss_r, g_r = U.loss_grad(p, *(a.astype(np.float64) for a in (x, d, t)), scales, q=q)
    assert abs(loss - loss_r) <= 1e-3 * abs(loss_r)
    o = 0
    for ci, co in LAYERS:
        for n in (27 * ci * co, co):
            assert rel_l2(g[o:o + n], g_r[o:o + n]) <= 3e-2
            o += n
    assert rel_l2(g[o:], g_r[o:]) <= 3e-2
