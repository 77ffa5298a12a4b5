"""Which kernel a convolution or a product takes on both sides of the split kernels' rules, and
its values.

The convolutions' rule compares estimated times (csrc/split.hip, conv_run): few input channels fill a matrix
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
    ((16, 512, 7, 7), (512, 512, 3, 3), 1, 1, True),   # 784 pixels: 112 / 59 us
    ((31, 64, 7, 7), (320, 64, 5, 5), 1, 2, True),     # 1519 pixels
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


def test_superpixel_2x2_beyond_1gib():
    """A 3x3 stride-2 dX of 1 GiB, which the split kernels don't take: sampled outputs of the 2x2
    super-pixel form."""
    import torch
    from katsu_amd import ops
    xs, ws = (4700, 16, 60, 60), (20, 16, 3, 3)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    gy = torch.randn((xs[0], ws[0], 29, 29), generator=gen, device="cuda")
    w = synth.he_normal(2, ws)
    wd, out = torch.from_numpy(w).cuda(), torch.empty(xs, device="cuda")
    call = lambda: ops.conv2d_backward_data(gy, wd, xs, 2, 0, out=out)
    assert kernels(call) == {"direct_fwd_kernel"}
    for n in (0, 2345, 4699):
        at = random_samples((1,) + xs[1:], 200, 5) + edge_samples((1,) + xs[1:])
        vals, sabs = sample_dx(gy[n:n + 1].cpu().numpy(), w, (1,) + xs[1:], 2, 0, at)
        got = out[n:n + 1].cpu().numpy()
        assert_within(np.array([got[i] for i in at]), vals, sabs, ws[0] * 9, f"image {n}")


GEMM_ROUTES = [  # m, k, n, kernel
    (2052, 16, 2100, "gemm_kernel"),     # short sums: 128-tiles
    (1000, 20, 1100, "gemm_kernel"),     # 64-tiles
    (33, 31, 65, "igemm_kernel"),        # unaligned and short
    (33, 32, 65, "split_gemm_kernel"),
    (512, 512, 512, "gemm_kernel"),      # 32-tiles
    (64, 904, 64, "gemm_kernel"),        # a long sum of few tiles: split over blocks
    (64, 900, 64, "split_gemm_kernel"),
    (1024, 1024, 1024, "gemm_rd_kernel"),
    (2048, 32, 2048, "split_gemm_kernel"),
]


@pytest.mark.parametrize("m,k,n,kernel", GEMM_ROUTES)
def test_gemm_route(m, k, n, kernel):
    import torch
    from katsu_amd import ops
    a, b = synth.uniform(1, (m, k)), synth.uniform(2, (k, n))
    ad, bd = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    out = torch.empty((m, n), device="cuda")
    assert kernel in kernels(lambda: ops.gemm(ad, bd, m, n, k, out=out))
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert_within(out.cpu().numpy(), a64 @ b64, np.abs(a64) @ np.abs(b64), k, "C")


VJP_ROUTES = [  # m, k, n, kernels: dA sums n products, dB m
    (240, 384, 16, {"gemm_vjp_kernel"}),  # one launch: 8.3 us, one product on each side 10.3
    (400, 56464, 4, {"gemm_kernel", "split_gemm_kernel"}),
    (64, 2048, 64, {"split_gemm_vjp_kernel"}),
]


@pytest.mark.parametrize("m,k,n,names", VJP_ROUTES)
def test_vjp_route(m, k, n, names):
    import torch
    from katsu_amd import ops
    a, b, g = (synth.uniform(i, s) for i, s in ((1, (m, k)), (2, (k, n)), (3, (m, n))))
    ad, bd, gd = (torch.from_numpy(v).cuda() for v in (a, b, g))
    da, db = torch.zeros_like(ad), torch.zeros_like(bd)
    assert kernels(lambda: ops.matmul_vjp(ad, bd, gd, da, db)) == names
    a64, b64, g64 = (v.astype(np.float64) for v in (a, b, g))
    assert_within(da.cpu().numpy(), g64 @ b64.T, np.abs(g64) @ np.abs(b64).T, n + 1, "dA")
    assert_within(db.cpu().numpy(), a64.T @ g64, np.abs(a64).T @ np.abs(g64), m + 1, "dB")
