"""The convolution kernels on the bf16 matrix cores (csrc/splitconv.hpp) against float64.

Layers at the edges of their tiles: images that share a tile and images that do not, strips of
wide rows, channel counts off the chunks of 16 and the tiles of 32 and 64, filters of fewer and
more taps than are staged together, both strides and all their phases, padding beyond the
filter.  Each test asserts that the split kernel is the one that runs.  Bound: that of a float32 dot product in any order (tests/parity.py); what the split
leaves out is at most a quarter of the rounding it counts per product."""
import numpy as np
import pytest

from katsu_amd import synth
from tests.parity import assert_within
from tests.routes import kernels

pytestmark = pytest.mark.gpu

LAYERS = [  # x, w, stride, pad
    ((3, 81, 7, 7), (33, 81, 3, 3), 1, 1),       # images share tiles, tails of every kind
    ((2, 40, 29, 31), (70, 40, 3, 3), 1, 1),
    ((1, 80, 20, 65), (32, 80, 3, 3), 1, 1),     # two strips of 33 and 32 columns
    ((2, 41, 12, 130), (20, 41, 5, 5), 1, 2),    # three strips, 25 taps
    ((32, 32, 40, 48), (64, 32, 3, 3), 1, 1),    # 64 x 256 and 32 x 256 tiles
    ((9, 24, 56, 56), (96, 24, 2, 3), 1, 0),     # rectangular filter, no padding
    ((2, 120, 13, 11), (18, 120, 3, 3), 1, 4),   # padding beyond the filter
    ((2, 50, 33, 47), (30, 50, 7, 7), 2, 3),     # stride 2: four phases of 16, 12, 12, 9 taps
    ((3, 36, 30, 29), (41, 36, 5, 5), 2, 2),
    ((2, 48, 21, 70), (40, 48, 4, 4), 2, 1),     # even filter
]


def _ref(x, w, gy, stride, pad):
    import torch
    t = [torch.from_numpy(v.astype(np.float64)) for v in (x, w, gy)]
    y = torch.nn.functional.conv2d(t[0], t[1], stride=stride, padding=pad)
    dx = torch.nn.grad.conv2d_input(x.shape, t[1], t[2], stride=stride, padding=pad)
    return y.numpy(), dx.numpy()


@pytest.mark.parametrize("xs,ws,stride,pad", LAYERS)
def test_split_conv(xs, ws, stride, pad):
    import torch
    from katsu_amd import ops
    x, w = synth.uniform(1, xs), synth.he_normal(2, ws)
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    gy = synth.normal(3, (xs[0], ws[0], oh, ow))
    dev = lambda a: torch.from_numpy(a).cuda()
    y, dx = _ref(x, w, gy, stride, pad)
    sy, sdx = _ref(np.abs(x), np.abs(w), np.abs(gy), stride, pad)
    kf, kb = ws[1] * ws[2] * ws[3], ws[0] * ws[2] * ws[3]
    xd, wd, gd = dev(x), dev(w), dev(gy)
    assert kernels(lambda: ops.conv2d_forward(xd, wd, stride, pad)) == {"split_conv_kernel"}
    assert kernels(lambda: ops.conv2d_backward_data(gd, wd, xs, stride,
                                                    pad)) == {"split_conv_kernel"}
    got = ops.conv2d_forward(xd, wd, stride, pad)
    assert_within(got.cpu().numpy(), y, sy, kf, "y")
    got = ops.conv2d_backward_data(gd, wd, xs, stride, pad)
    assert_within(got.cpu().numpy(), dx, sdx, kb, "dX")
    old = synth.uniform(4, xs)
    acc = dev(old)
    ops.conv2d_backward_data(dev(gy), dev(w), xs, stride, pad, out=acc, beta=1.0)
    assert_within(acc.cpu().numpy(), old + dx, np.abs(old) + sdx, kb + 1, "dX, beta 1")
    # Twice the same bits, and the same as the one-call backward's.
    dx2, _ = ops.conv2d_backward(dev(x), dev(w), dev(gy), stride, pad)
    assert torch.equal(dx2, got)


@pytest.mark.parametrize("xs,ws,stride,pad", [LAYERS[0], LAYERS[3], LAYERS[8]])
def test_split_conv_nonfinite(xs, ws, stride, pad):
    """Inf and NaN reach exactly the outputs whose visited taps hold them (padding and the
    filter's missing taps multiply nothing)."""
    import torch
    from katsu_amd import ops
    x, w = synth.uniform(1, xs), synth.he_normal(2, ws)
    x[0, 0, 0, 0], x[-1, 1, -1, -1], x[0, -1, xs[2] // 2, xs[3] // 2] = np.inf, -np.inf, np.nan
    y = ops.conv2d_forward(torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), stride,
                           pad).cpu().numpy()
    xd, wd = x.astype(np.float64), w.astype(np.float64)
    ref = np.zeros(y.shape)
    h, wdt = xs[2], xs[3]
    with np.errstate(invalid="ignore"):
        for oy in range(y.shape[2]):
            for ox in range(y.shape[3]):
                y0, x0 = oy * stride - pad, ox * stride - pad
                r = slice(max(0, -y0), min(ws[2], h - y0))
                s = slice(max(0, -x0), min(ws[3], wdt - x0))
                patch = xd[:, :, y0 + r.start:y0 + r.stop, x0 + s.start:x0 + s.stop]
                ref[:, :, oy, ox] = (patch[:, None] * wd[None, :, :, r, s]).sum((2, 3, 4))
    for mask in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(mask(y), mask(ref))
    assert np.isfinite(ref).any() and not np.isfinite(ref).all()


@pytest.mark.parametrize("xs,ws,stride,pad", [LAYERS[0], LAYERS[3], LAYERS[8]])
def test_split_dx_nonfinite(xs, ws, stride, pad):
    """The same of the data gradient, at stride 2 in all four phases."""
    import torch
    from katsu_amd import ops
    w = synth.he_normal(2, ws)
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    gy = synth.normal(3, (xs[0], ws[0], oh, ow))
    gy[0, 0, 0, 0], gy[-1, 1, -1, -1], gy[0, -1, oh // 2, ow // 2] = np.inf, -np.inf, np.nan
    w[2, 3, 0, 0] = np.inf
    dx = ops.conv2d_backward_data(torch.from_numpy(gy).cuda(), torch.from_numpy(w).cuda(), xs,
                                  stride, pad).cpu().numpy()
    gd, wd = gy.astype(np.float64), w.astype(np.float64)
    ref = np.zeros(xs)
    with np.errstate(invalid="ignore"):
        for oy in range(oh):
            for ox in range(ow):
                y0, x0 = oy * stride - pad, ox * stride - pad
                r = slice(max(0, -y0), min(ws[2], xs[2] - y0))
                s = slice(max(0, -x0), min(ws[3], xs[3] - x0))
                ref[:, :, y0 + r.start:y0 + r.stop, x0 + s.start:x0 + s.stop] += (
                    gd[:, :, oy, ox][:, :, None, None, None] * wd[None, :, :, r, s]).sum(1)
    for mask in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(mask(dx), mask(ref))
    assert np.isfinite(ref).any() and not np.isfinite(ref).all()


DW_LAYERS = [  # x, w, stride, pad: 1.5 GFLOP or more, so that the split kernel takes them
    ((30, 96, 20, 20), (128, 96, 3, 3), 1, 1),   # whole images
    ((40, 160, 14, 14), (130, 160, 3, 3), 1, 1),  # tiles across images, channel tail
    ((3, 40, 90, 130), (60, 40, 5, 5), 1, 2),    # strips, three sets of taps
    ((8, 64, 30, 33), (64, 64, 7, 7), 1, 3),
    ((40, 64, 199, 15), (64, 64, 3, 2), 2, 1),   # stride 2: few columns, whose rows fit the LDS
]


@pytest.mark.parametrize("xs,ws,stride,pad", DW_LAYERS)
def test_split_dw(xs, ws, stride, pad):
    """Sampled exact sums, the corners among them; the same bits twice and in the one-call
    backward; beta = 1; and Inf and NaN in the sums that hold them only."""
    import torch
    from katsu_amd import ops
    from tests.parity import random_samples, sample_dw
    x, w = synth.uniform(1, xs), synth.he_normal(2, ws)
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    gy = synth.normal(3, (xs[0], ws[0], oh, ow))
    dev = lambda a: torch.from_numpy(a).cuda()
    at = random_samples(ws, 200, 5) + [(0, 0, 0, 0), tuple(d - 1 for d in ws)]
    pick = lambda t: np.array([t[i] for i in at])
    ref, sabs = sample_dw(x, gy, ws, stride, pad, at)
    n = xs[0] * oh * ow
    xd, gd = dev(x), dev(gy)
    assert "split_dw_kernel" in kernels(
        lambda: ops.conv2d_backward_filter(xd, gd, ws, stride, pad))
    dw = ops.conv2d_backward_filter(xd, gd, ws, stride, pad)
    assert_within(pick(dw.cpu().numpy()), ref, sabs, n, "dW")
    _, dw2 = ops.conv2d_backward(dev(x), dev(w), dev(gy), stride, pad)
    assert torch.equal(dw, dw2)
    old = synth.uniform(4, ws)
    acc = dev(old)
    ops.conv2d_backward_filter(dev(x), dev(gy), ws, stride, pad, out=acc, beta=1.0)
    assert torch.equal(acc, dev(old) + dw)
    # One pixel of one input channel, at a corner: only the taps that reach it.
    x[1, 2, 0, 0] = np.inf
    gy[1, 3, 0, 0] = 0.5
    got = ops.conv2d_backward_filter(dev(x), dev(gy), ws, stride, pad).cpu().numpy()
    bad = ~np.isfinite(got)
    reach = np.zeros(ws[2:], bool)
    for i in range(ws[2]):
        for j in range(ws[3]):
            oy, ox = (pad - i) / stride, (pad - j) / stride
            reach[i, j] = oy in range(oh) and ox in range(ow)
    assert np.array_equal(bad[3, 2], reach) and not np.delete(bad, 2, axis=1).any()


def test_split_conv_large_planes():
    """Channels far apart: a chunk after the two of 17 channels would end beyond 2^31 bytes, and
    the tensors end just below 1 GiB.  Sampled outputs, corners and both passes."""
    import torch
    from katsu_amd import ops
    xs, ws, hw = (1, 17, 3400, 3400), (20, 17, 3, 3), 3400
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    x = torch.randn(xs, generator=gen, device="cuda")
    gy = torch.randn((1, 20, hw, hw), generator=gen, device="cuda")
    w = torch.from_numpy(synth.he_normal(2, ws)).cuda()
    rng = np.random.default_rng(4)
    at = [tuple(p) for p in rng.integers(0, hw, (60, 2))] + [(0, 0), (hw - 1, hw - 1), (0, hw - 1)]

    def check(got, inp, filt, what):
        for y0, x0 in at:
            r0, c0 = max(0, y0 - 1), max(0, x0 - 1)
            patch = inp[0, :, r0:y0 + 2, c0:x0 + 2].double()
            f = filt[:, :, r0 - y0 + 1:r0 - y0 + 1 + patch.shape[1],
                     c0 - x0 + 1:c0 - x0 + 1 + patch.shape[2]].double()
            ref = (patch * f).sum((1, 2, 3)).cpu().numpy()
            sab = (patch.abs() * f.abs()).sum((1, 2, 3)).cpu().numpy()
            assert_within(got[0, :, y0, x0].cpu().numpy(), ref, sab, inp.shape[1] * 9,
                          f"{what} at {y0}, {x0}")

    check(ops.conv2d_forward(x, w, 1, 1), x, w, "y")
    check(ops.conv2d_backward_data(gy, w, xs, 1, 1), gy, w.transpose(0, 1).flip(2, 3), "dX")
