"""fp32 models with few rows whose K is no whole number of k-groups, or whose rows are not 16-byte aligned: the 16-column
VALU kernel (up to 4 rows, mnb_gemv.hip) and the 16-row kernel on the fp32 matrix cores (mnb_rows16_f32.hip), against the
CPU oracle.  What lies behind the last element of a row is NaN: reading it into a sum would show."""
import numpy as np
import pytest
import torch

from gpu_util import check_against_oracle, dev, make_op
from onnxruntime_amd import _lib
from onnxruntime_amd.synthetic import make_case

pytestmark = pytest.mark.gpu


# K: the shortest, one to three elements beyond a piece of four, beyond a k-group, beyond a chunk, beyond 2048 staged k
@pytest.mark.parametrize("K", [4, 5, 31, 33, 100, 126, 130, 1532, 2051, 3652])
@pytest.mark.parametrize("bits,bs,zp", [(4, 32, True), (4, 16, False), (8, 128, True), (2, 64, True)])
def test_ragged_k(oracle, bits, bs, zp, K):
    for M, N in ((1, 70), (3, 12300), (4, 500), (5, 40), (17, 300), (64, 1000), (2, 100000), (7, 100001), (137, 300), (900, 70)):
        if N * K > 4e6:
            continue
        c = make_case(M, N, K, bits, bs, np.float32, has_zp=zp, has_bias=M % 2 == 1, seed=M + N + K)
        op = make_op(c)
        for pitch, first in ((K, 0), (K + 3, 1)):
            store = torch.full((first + M * pitch + 8,), float("nan"), device="cuda")
            a = store[first:first + M * pitch].view(M, pitch)[:, :K]
            a.copy_(dev(c.A))
            y = op.Compute(a, bias=dev(c.bias))
            check_against_oracle(oracle, c, y.cpu().numpy())


@pytest.mark.parametrize("bits,bs", [(4, 128), (4, 16), (8, 32), (2, 64)])
@pytest.mark.parametrize("M,N,K", [(1, 70, 130), (2, 500, 1275), (4, 40, 4101), (9, 300, 1275)])
def test_activations_whose_block_sums_lie_beyond_fp32(oracle, bits, bs, M, N, K):
    """A sum of a block's products before its scale would overflow; the result does not."""
    c = make_case(M, N, K, bits, bs, np.float32, has_zp=True, seed=K)
    c.A = (c.A * np.float32(2.0) ** 121).astype(np.float32)
    c.scales = np.abs(c.scales) * np.float32(2.0 ** -10)
    y = make_op(c).Compute(dev(c.A)).cpu().numpy()
    assert np.isfinite(y).all()
    check_against_oracle(oracle, c, y)


def test_whole_k_with_rows_that_are_not_aligned(oracle):
    for M in (2, 9, 40):
        c = make_case(M, 200, 512, 4, 32, np.float32, has_zp=True, seed=M)
        a = torch.full((M, 515), float("nan"), device="cuda")[:, 1:513]
        a.copy_(dev(c.A))
        check_against_oracle(oracle, c, make_op(c).Compute(a).cpu().numpy())


def test_the_kernels_that_take_them():
    name = lambda M, N, K: _lib.load().MnbGemmKernelName(M, N, K, 4, 32, _lib.DTYPE_FLOAT)  # noqa: E731
    assert name(4, 500, 1532) == b"mnb_gemv_kernel"
    assert name(5, 500, 1532) == b"mnb_rows16_f32_ragged_kernel"
    assert name(64, 300, 130) == b"mnb_rows16_f32_ragged_kernel"
    assert name(137, 70, 856) == b"mnb_rows16_f32_ragged_kernel"
    assert name(137, 70, 856 - 300) == b"mnb_rows16_f32_ragged_kernel"
    assert name(137, 70, 130) == b"mnb_rows16_f32_ragged_kernel"
    # many columns of short K: little work for each of its workgroups
    assert name(782, 2365, 47) == name(72, 13422, 17) == name(55, 23486, 10) == name(17, 28000, 5) == b"mnb_gemm32_kernel"
    assert name(5, 500, 3) == b"mnb_gemm_generic_kernel"
    # wide matrices of short K, and more columns than a launch of the others holds
    for M, N, K in ((1, 300000, 33), (4, 131072, 65), (8, 300000, 65), (1, 70 << 20, 1023), (9, 70 << 20, 1023)):
        assert name(M, N, K) == b"mnb_gemm_generic_kernel"
    assert name(1, 32768, 65) == name(4, 28672, 130) == b"mnb_gemv_kernel"
    assert name(8, 65536, 65) == name(16, 300000, 1023) == b"mnb_rows16_f32_ragged_kernel"
