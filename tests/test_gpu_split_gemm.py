"""The GEMM on the bf16 matrix cores (csrc/splitgemm.hpp) against float64.

Shapes at the edges of each of its tiles (32, 64, 128 and 256 x 128), with sums that end
inside a matrix step, a stage and a run of 128 k, from pointers that are only 4-byte aligned;
forward, both VJP products (in one launch or two), and beta = 1.  Bound: that of a float32 dot
product in any order (tests/parity.py); the split's own error, at most 2^-26 of each product, is
a quarter of the rounding it counts per product.  Whole numbers of 12 by 4 bits are exact in two
of the six bf16 products (tests/test_gpu_split_precision.py has numbers for each of them)."""
import numpy as np
import pytest

from katsu_amd import synth
from tests.parity import assert_within
from tests.routes import kernels

pytestmark = pytest.mark.gpu

SHAPES = [  # m, k, n; the tile of the forward product
    (31, 40, 33), (65, 129, 64), (48, 33, 56), (17, 700, 23),  # 32
    (1001, 100, 777), (640, 333, 641),                         # 64
    (1500, 47, 1501),                                          # 128
    (2049, 161, 2040),                                         # 256 x 128
]


def _dev(a, shift=0):
    """The array on the GPU, `shift` floats past an aligned address."""
    import torch
    buf = torch.empty(a.size + shift, device="cuda", dtype=torch.float32)
    t = buf[shift:].view(a.shape)
    t.copy_(torch.from_numpy(a))
    return t


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("shift", [0, 1])
def test_split_gemm(m, k, n, shift):
    from katsu_amd import ops
    a, b, g = (synth.uniform(s, sh) for s, sh in ((11, (m, k)), (12, (k, n)), (13, (m, n))))
    ad, bd, gd = (_dev(v, shift) for v in (a, b, g))
    a64, b64, g64 = (v.astype(np.float64) for v in (a, b, g))
    c = _dev(np.full((m, n), np.nan, np.float32), shift)
    assert kernels(lambda: ops.gemm(ad, bd, m, n, k, out=c)) == {"split_gemm_kernel"}
    assert_within(c.cpu().numpy(), a64 @ b64, np.abs(a64) @ np.abs(b64), k, "C")
    da0, db0 = synth.uniform(14, (m, k)), synth.uniform(15, (k, n))
    da, db = _dev(da0, shift), _dev(db0, shift)
    ops.matmul_vjp(ad, bd, gd, da, db)
    assert_within(da.cpu().numpy(), da0 + g64 @ b64.T,
                  np.abs(da0) + np.abs(g64) @ np.abs(b64).T, n + 1, "dA")
    assert_within(db.cpu().numpy(), db0 + a64.T @ g64,
                  np.abs(db0) + np.abs(a64).T @ np.abs(g64), m + 1, "dB")


@pytest.mark.parametrize("m,k,n", SHAPES[::2])
def test_split_gemm_integers_exact(m, k, n):
    """Operands of up to 12 bits (two bf16 parts): every sum stays below 2^24 in steps of one."""
    from katsu_amd import ops
    rng = np.random.default_rng(5)
    a = rng.integers(-3000, 3001, (m, k)).astype(np.float32)
    b = rng.integers(-7, 8, (k, n)).astype(np.float32)
    c = ops.gemm(_dev(a), _dev(b), m, n, k).cpu().numpy()
    assert np.array_equal(c, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32))


@pytest.mark.parametrize("m,k,n", SHAPES[1::2])
def test_split_gemm_nonfinite(m, k, n):
    """A tile with a non-finite value is computed again in float32: same NaN and Inf as numpy's
    sums, also from a value that rounds to Inf in bf16."""
    from katsu_amd import ops
    a, b = synth.uniform(11, (m, k)), synth.uniform(12, (k, n))
    a[0, 0], a[m - 1, k - 1], b[k // 2, n - 1] = np.inf, np.nan, -np.inf
    a[m // 2, 1], b[1, :] = np.finfo(np.float32).max, 0.25
    with np.errstate(invalid="ignore"):
        ref = a.astype(np.float64) @ b.astype(np.float64)
    got = ops.gemm(_dev(a), _dev(b), m, n, k).cpu().numpy()
    for mask in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(mask(got), mask(ref))
    fin = np.isfinite(ref)
    s = np.abs(np.where(np.isfinite(a), a, 0)).astype(np.float64) @ np.abs(
        np.where(np.isfinite(b), b, 0)).astype(np.float64)
    assert_within(got[fin], ref[fin], s[fin], k, "C")
