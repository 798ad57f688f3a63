"""fp32 models with many rows: activations split into three bfloat16 parts (mnb_gemm32_split.hip), against the oracle.

A block's sum takes at most 6 matrix instructions of 16 products each, every addition rounding by at most 2^-23 of what
has been summed, and the blocks' sums are joined by at most K / 32 + 8 more: |err| <= (K / 32 + 110) 2^-23 sum |a w|."""
import numpy as np
import pytest

from gpu_util import dev, make_op
from onnxruntime_amd import _lib
from onnxruntime_amd.synthetic import make_case

pytestmark = pytest.mark.gpu


def run(c):
    need = _lib.load().MnbGemmWorkspaceSize(c.M, c.N, c.K, c.bits, c.block_size, int(c.zero_points is not None),
                                            _lib.DTYPE_FLOAT)
    assert need >= c.M * c.K * 6  # the split activations: this kernel serves the shape
    return make_op(c).Compute(dev(c.A), bias=dev(c.bias)).cpu().numpy()


# rows of the workgroup's tile: 32 (every step its own team), 64, 128, 256; ragged rows, columns and steps of every size
@pytest.mark.parametrize("M,N,K", [(97, 4096, 4096), (200, 4090, 1056), (513, 4090, 544), (990, 4090, 992),
                                   (230, 28600, 260)])
@pytest.mark.parametrize("bits,bs,zp,bias", [(4, 32, True, True), (4, 16, True, False), (4, 128, False, False),
                                             (8, 64, True, True), (8, 16, False, True), (2, 32, False, False)])
def test_parity(oracle, M, N, K, bits, bs, zp, bias):
    c = make_case(M, N, K, bits, bs, np.float32, has_zp=zp, has_bias=bias, seed=M + bits)
    c.A *= np.exp2(np.random.default_rng(1).integers(-20, 20, size=(M, 1))).astype(np.float32)
    y = run(c)
    rows = np.unique([0, 1, 31, 32, 63, 64, 96, 128, 255, 256, M - 2, M - 1])
    rows = rows[rows < M]
    want, bound = oracle.C.matmul_f64(c.A[rows], c.B, c.scales, c.zero_points, c.bias, N, K, bits, bs, nthreads=8)
    assert np.all(np.abs(y[rows] - want) <= (K / 32 + 110) * 2.0**-23 * bound)


def test_infinities_nans_and_extreme_values(oracle):
    """The parts of an infinity or a NaN are itself and zeros; the smallest and largest numbers keep all their bits."""
    c = make_case(200, 4096, 1024, 4, 32, np.float32, has_zp=True, seed=2)
    c.A[:] = 0
    c.A[0, 5], c.A[1, 6], c.A[2, 7] = np.inf, -np.inf, np.nan
    c.A[3, 8], c.A[4, 9], c.A[5, 10] = 3e34, 1.0000001e-30, np.float32(1) + np.float32(2)**-23
    y = run(c)
    w = oracle.C.dequantize(c.B, c.scales, c.zero_points, c.N, c.K, 4, 32)
    with np.errstate(invalid="ignore"):
        for r, k in enumerate(range(5, 11)):
            want = c.A[r, k] * w[:, k]
            assert np.array_equal(np.isnan(y[r]), np.isnan(want))
            fine = np.isfinite(want)
            assert np.array_equal(y[r][~fine & ~np.isnan(want)], want[~fine & ~np.isnan(want)])
            np.testing.assert_allclose(y[r][fine], want[fine], rtol=2.0**-21)
    assert not y[6:].any()
