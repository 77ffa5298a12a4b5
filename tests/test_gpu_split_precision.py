"""What the three bf16 values and the six products of csrc/split3.hpp must keep of a float32.

The bound of tests/parity.py is relative to each operand, whatever its size: it also holds
where an operand is so small that bf16 values of it would be subnormal, or so large that a
scaled one overflows.  It grows with the length of the sum, though, and the loss of a whole
product would stay inside it: bounds on the 2-norm and sums that a single product decides
hold the six to account."""
import numpy as np
import pytest

from katsu_amd import synth
from tests.parity import assert_within, random_samples, sample_dw, sample_dx, sample_fwd
from tests.test_gpu_split_conv import DW_LAYERS, LAYERS
from tests.test_gpu_split_gemm import SHAPES, _dev

pytestmark = pytest.mark.gpu

# Operand sizes: normal floats near the smallest, subnormal ones, and large ones, with a
# partner that brings the products back to ordinary numbers.
SCALES = [(1e-34, 1e15), (1e-37, 1e20), (1e20, 1e-37), (1e-40, 1e25), (1e-18, 1e-18),
          (1e33, 1e-30), (1e20, 1e14)]


def _scaled(seed, shape, s):
    return (synth.uniform(seed, shape).astype(np.float64) * s).astype(np.float32)


def _rel(got, ref):
    """Error in the 2-norm."""
    return float(np.linalg.norm(got.cpu().numpy() - ref) / np.linalg.norm(ref))


def _pick(t, at):
    v = t.cpu().numpy()
    return np.array([v[i] for i in at])


@pytest.mark.parametrize("m,k,n", SHAPES[::2] + SHAPES[5:6] + SHAPES[7:])
@pytest.mark.parametrize("s,t", SCALES)
def test_gemm_operand_scales(m, k, n, s, t):
    from katsu_amd import ops
    a, b = _scaled(11, (m, k), s), _scaled(12, (k, n), t)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    c = ops.gemm(_dev(a), _dev(b), m, n, k).cpu().numpy()
    assert_within(c, a64 @ b64, np.abs(a64) @ np.abs(b64), k, "C")


@pytest.mark.parametrize("xs,ws,stride,pad", [LAYERS[0], LAYERS[4], LAYERS[7]])
@pytest.mark.parametrize("s,t", SCALES)
def test_conv_operand_scales(xs, ws, stride, pad, s, t):
    from katsu_amd import ops
    x, w = _scaled(1, xs, s), _scaled(2, ws, t)
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    gs = (xs[0], ws[0], oh, ow)
    gy = _scaled(3, gs, s)
    y = ops.conv2d_forward(_dev(x), _dev(w), stride, pad)
    at = random_samples(gs, 300, 7)
    assert_within(_pick(y, at), *sample_fwd(x, w, stride, pad, at), ws[1] * ws[2] * ws[3], "y")
    dx = ops.conv2d_backward_data(_dev(gy), _dev(w), xs, stride, pad)
    at = random_samples(xs, 300, 8)
    assert_within(_pick(dx, at), *sample_dx(gy, w, xs, stride, pad, at), ws[0] * ws[2] * ws[3],
                  "dX")


@pytest.mark.parametrize("s,t", SCALES)
def test_dw_operand_scales(s, t):
    from katsu_amd import ops
    xs, ws, stride, pad = DW_LAYERS[1]
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    x, gy = _scaled(1, xs, s), _scaled(3, (xs[0], ws[0], oh, ow), t)
    dw = ops.conv2d_backward_filter(_dev(x), _dev(gy), ws, stride, pad)
    at = random_samples(ws, 200, 5)
    assert_within(_pick(dw, at), *sample_dw(x, gy, ws, stride, pad, at), xs[0] * oh * ow, "dW")


# Sums of long runs on the matrix cores lose the tails of terms of one sign, so the kernels
# break them: the error must not grow with the filter.  Bounds on the 2-norm, in roundings of
# the total (2^-24 = 6e-8): 2.5 for terms of one sign, 6 for signed ones, whose result is
# smaller than its terms.  Sums over all taps of a chunk showed 3.0e-7 and 4.3e-7.
LONG_FILTERS = [  # x, w, stride, pad
    ((4, 12, 45, 52), (128, 12, 7, 7), 1, 3),    # 49 taps in one chunk, one wave for all
    ((2, 16, 40, 40), (64, 16, 15, 15), 1, 7),   # 225 taps
    ((8, 15, 33, 31), (40, 15, 5, 5), 1, 2),
    ((2, 32, 56, 56), (64, 32, 3, 3), 1, 1),
]


@pytest.mark.parametrize("xs,ws,stride,pad", LONG_FILTERS)
@pytest.mark.parametrize("one_signed", [True, False])
def test_conv_error_does_not_grow_with_the_filter(xs, ws, stride, pad, one_signed):
    from katsu_amd import ops
    from tests.test_gpu_split_conv import _ref
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    x, w, gy = (synth.uniform(s, sh) for s, sh in ((1, xs), (2, ws), (3, (xs[0], ws[0], oh, ow))))
    if one_signed:
        x, w, gy = np.abs(x), np.abs(w), np.abs(gy)
    y, dx = _ref(x, w, gy, stride, pad)
    lim = 1.5e-7 if one_signed else 3.5e-7
    err_y = _rel(ops.conv2d_forward(_dev(x), _dev(w), stride, pad), y)
    err_dx = _rel(ops.conv2d_backward_data(_dev(gy), _dev(w), xs, stride, pad), dx)
    assert max(err_y, err_dx) < lim, (err_y, err_dx)


# The error in the 2-norm of sums of uniform numbers of both signs is 4e-9 for the six products
# with nothing rounded and 2.0e-6 (in float64, whatever the length) without the smallest of them;
# the float32 total adds a rounding of 6e-8 to each of a few partial sums.
SIX_PRODUCTS = 5e-7


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
def test_gemm_two_norm(m, k, n, ta, tb):
    from katsu_amd import ops
    a, b = synth.uniform(21, (m, k)), synth.uniform(22, (k, n))
    ad, bd = _dev(np.ascontiguousarray(a.T) if ta else a), _dev(np.ascontiguousarray(b.T) if tb else b)
    c = ops.gemm(ad, bd, m, n, k, trans_a=ta, trans_b=tb)
    assert _rel(c, a.astype(np.float64) @ b.astype(np.float64)) < SIX_PRODUCTS


@pytest.mark.parametrize("xs,ws,stride,pad", LAYERS)
def test_conv_two_norm(xs, ws, stride, pad):
    from katsu_amd import ops
    from tests.test_gpu_split_conv import _ref
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    x, w, gy = (synth.uniform(s, sh) for s, sh in ((1, xs), (2, ws), (3, (xs[0], ws[0], oh, ow))))
    y, dx = _ref(x, w, gy, stride, pad)
    assert _rel(ops.conv2d_forward(_dev(x), _dev(w), stride, pad), y) < SIX_PRODUCTS
    assert _rel(ops.conv2d_backward_data(_dev(gy), _dev(w), xs, stride, pad), dx) < SIX_PRODUCTS


@pytest.mark.parametrize("xs,ws,stride,pad", DW_LAYERS)
def test_dw_two_norm(xs, ws, stride, pad):
    from katsu_amd import ops
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    x, gy = synth.uniform(1, xs), synth.uniform(3, (xs[0], ws[0], oh, ow))
    at = random_samples(ws, 200, 5)
    ref, _ = sample_dw(x, gy, ws, stride, pad, at)
    got = _pick(ops.conv2d_backward_filter(_dev(x), _dev(gy), ws, stride, pad), at)
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < SIX_PRODUCTS


# Whole numbers of 24 bits times powers of two need all three parts of the one operand, and of 12
# by 12 bits both parts of each: with one such product a sum, the result is exact or wrong.
KINDS = ["24 bits left", "24 bits right", "12 bits each"]


def _parts(kind, left, right):
    """Operands of the two shapes, odd or a power of two."""
    rng = np.random.default_rng(31)
    odd = lambda bits, shape: (2 * rng.integers(2 ** (bits - 2), 2 ** (bits - 1), shape) + 1) * \
        rng.choice([-1, 1], shape)
    two = lambda shape: 2.0 ** rng.integers(-8, 9, shape)
    a, b = {"24 bits left": lambda: (odd(24, left), two(right)),
            "24 bits right": lambda: (two(left), odd(24, right)),
            "12 bits each": lambda: (odd(12, left), odd(12, right))}[kind]()
    return a.astype(np.float32), b.astype(np.float32)


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("kind", KINDS)
def test_gemm_each_product(m, k, n, kind):
    from katsu_amd import ops
    col, b = _parts(kind, (m,), (k, n))
    a = np.zeros((m, k), np.float32)
    at = np.arange(m) * 7 % k
    a[np.arange(m), at] = col
    ref = col[:, None].astype(np.float64) * b[at]
    for ta, tb in ((False, False), (False, True), (True, False)):
        c = ops.gemm(_dev(np.ascontiguousarray(a.T) if ta else a),
                     _dev(np.ascontiguousarray(b.T) if tb else b), m, n, k, trans_a=ta, trans_b=tb)
        assert np.array_equal(c.cpu().numpy(), ref), (ta, tb)


@pytest.mark.parametrize("xs,ws,stride,pad", LAYERS)
@pytest.mark.parametrize("kind", KINDS)
def test_conv_each_product(xs, ws, stride, pad, kind):
    """One filter value per output channel (forward) or per input channel of the first output
    channel (data gradient)."""
    from katsu_amd import ops
    from tests.test_gpu_split_conv import _ref
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    gs = (xs[0], ws[0], oh, ow)
    K, C, R, S = ws
    w, wb = np.zeros(ws, np.float32), np.zeros(ws, np.float32)
    i, j = np.arange(K), np.arange(C)
    x, w[i, i * 5 % C, i % R, i * 3 % S] = _parts(kind, xs, (K,))
    gy = np.zeros(gs, np.float32)
    gy[:, 0], wb[0, j, j % R, j * 3 % S] = _parts(kind, (xs[0], oh, ow), (C,))
    y, _ = _ref(x, w, gy, stride, pad)
    _, dx = _ref(x, wb, gy, stride, pad)
    assert np.array_equal(ops.conv2d_forward(_dev(x), _dev(w), stride, pad).cpu().numpy(), y)
    got = ops.conv2d_backward_data(_dev(gy), _dev(wb), xs, stride, pad)
    assert np.array_equal(got.cpu().numpy(), dx)


@pytest.mark.parametrize("xs,ws,stride,pad", DW_LAYERS)
@pytest.mark.parametrize("kind", KINDS)
def test_dw_each_product(xs, ws, stride, pad, kind):
    """One gradient pixel per output channel."""
    from katsu_amd import ops
    oh, ow = ((xs[i + 2] + 2 * pad - ws[i + 2]) // stride + 1 for i in (0, 1))
    gy = np.zeros((xs[0], ws[0], oh, ow), np.float32)
    k = np.arange(ws[0])
    n, oy, ox = k * 11 % xs[0], k * 5 % oh, k * 3 % ow
    x, g = _parts(kind, xs, k.shape)
    gy[n, k, oy, ox] = g
    got = ops.conv2d_backward_filter(_dev(x), _dev(gy), ws, stride, pad).cpu().numpy()
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
    for i in k:
        y0, x0 = oy[i] * stride, ox[i] * stride
        ref = g[i] * xp[n[i], :, y0:y0 + ws[2], x0:x0 + ws[3]]
        assert np.array_equal(got[i], ref), i
