"""Which kernel a convolution takes on both sides of the split kernels' rule, and its values.

The rule compares estimated times (csrc/split.hip, conv_run): few input channels fill a matrix
step of 16, and few output channels a tile of 32, too little to pay for six bf16 products."""
import numpy as np
import pytest

from katsu_amd import synth
from tests.parity import assert_within, edge_samples, random_samples, sample_dx, sample_fwd
from tests.routes import kernels

pytestmark = pytest.mark.gpu

ROUTES = [  # pass, x, w, stride, pad, kernel; with the times of the generic or direct and the split one
    ("fwd", (2, 64, 56, 56), (64, 64, 3, 3), 1, 1, "split_conv_kernel"),
    ("fwd", (6, 3, 198, 154), (64, 3, 3, 3), 1, 0, "igemm_kernel"),     # 21 / 33 us
    ("fwd", (10, 2, 167, 141), (128, 2, 4, 4), 2, 1, "igemm_kernel"),   # 18 / 74 us
    ("fwd", (61, 24, 85, 112), (128, 24, 3, 3), 2, 0, "igemm_kernel"),  # 113 / 213 us
    ("fwd", (14, 5, 134, 107), (96, 5, 7, 7), 2, 3, "igemm_kernel"),    # 58 / 168 us
    ("dx", (20, 3, 196, 196), (16, 3, 7, 7), 2, 3, "direct_fwd_kernel"),
    ("dx", (59, 16, 74, 49), (1, 16, 3, 3), 1, 3, "igemm_kernel"),      # 10 / 23 us
    ("dx", (32, 64, 28, 28), (128, 64, 3, 3), 2, 0, "split_conv_kernel"),
    ("dx", (8, 96, 27, 27), (128, 96, 5, 5), 1, 2, "split_conv_kernel"),
]


@pytest.mark.parametrize("op,xs,ws,stride,pad,kernel", ROUTES)
def test_conv_route(op, xs, ws, stride, pad, kernel):
    import torch
    from katsu_amd import ops
    w = synth.he_normal(2, ws)
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    gs = (xs[0], ws[0], oh, ow)
    a = synth.uniform(1, xs if op == "fwd" else gs)
    ad, wd = torch.from_numpy(a).cuda(), torch.from_numpy(w).cuda()
    out = torch.empty(gs if op == "fwd" else xs, device="cuda")
    if op == "fwd":
        call = lambda: ops.conv2d_forward(ad, wd, stride, pad, out=out)
        ref, kred = sample_fwd, ws[1] * ws[2] * ws[3]
    else:
        call = lambda: ops.conv2d_backward_data(ad, wd, xs, stride, pad, out=out)
        ref, kred = (lambda a, w, st, p, at: sample_dx(a, w, xs, st, p, at)), ws[0] * ws[2] * ws[3]
    assert kernels(call) == {kernel}
    at = random_samples(out.shape, 200, 5) + edge_samples(out.shape)
    got = out.cpu().numpy()
    vals, sabs = ref(a, w, stride, pad, at)
    assert_within(np.array([got[i] for i in at]), vals, sabs, kred, op)


DW_ROUTES = [  # x, w, stride, pad, split or not, with the times of the float32 and the split kernel
    ((30, 96, 20, 20), (128, 96, 3, 3), 1, 1, True),
    ((14, 96, 144, 80), (64, 96, 1, 1), 1, 1, False),  # one tap of nine: 47 / 88 us
    ((30, 16, 109, 119), (64, 16, 2, 2), 1, 0, False),  # 52 / 94 us
    ((3, 427, 9, 9), (384, 427, 5, 5), 1, 2, False),   # 243 pixels: 35 / 79 us
    ((5, 303, 10, 10), (234, 303, 7, 7), 1, 3, False),  # 500 pixels: 61 / 88 us
]


@pytest.mark.parametrize("xs,ws,stride,pad,split", DW_ROUTES)
def test_dw_route(xs, ws, stride, pad, split):
    import torch
    from katsu_amd import ops
    from tests.parity import sample_dw
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    x, gy = synth.uniform(1, xs), synth.normal(3, (xs[0], ws[0], oh, ow))
    xd, gd = torch.from_numpy(x).cuda(), torch.from_numpy(gy).cuda()
    out = torch.empty(ws, device="cuda")
    names = kernels(lambda: ops.conv2d_backward_filter(xd, gd, ws, stride, pad, out=out))
    assert ("split_dw_kernel" in names) == split, names
    at = random_samples(ws, 100, 5) + [(0, 0, 0, 0), tuple(d - 1 for d in ws)]
    got = out.cpu().numpy()
    vals, sabs = sample_dw(x, gy, ws, stride, pad, at)
    assert_within(np.array([got[i] for i in at]), vals, sabs, xs[0] * oh * ow, "dW")
