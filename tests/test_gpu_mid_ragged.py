"""The streaming kernel (mnb_mid.hip) on K that is a multiple of 8 but not of its chunks (128 with 4-bit weights, 64 with
8-bit), activations read in place: the pieces of the last chunk beyond K must not count, whatever lies there.

A lies in a wider matrix whose other columns are NaN; the last row ends with the allocation.  Gate of the 16-bit routes:
relative L2 <= 5e-3 against a float64 product over the reference dequantiser's W."""
import numpy as np
import pytest
import torch

from onnxruntime_amd import MatMulNBits, _lib
from onnxruntime_amd.synthetic import make_case

pytestmark = pytest.mark.gpu


# K: one piece in all, one piece beyond a chunk, one short of a chunk, a real one; N: one tile and ragged; rows: decode
# rows, partial and whole row tiles of both sizes
@pytest.mark.parametrize("K", [8, 136, 248, 2880])
@pytest.mark.parametrize("N,M", [(32, 1), (300, 16), (1000, 17), (5003, 37), (2880, 64), (300, 200)])
@pytest.mark.parametrize("bits,bs,zp", [(4, 32, True), (4, 16, False), (4, 128, True), (8, 64, True), (2, 32, False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_pieces_beyond_k(oracle, K, N, M, bits, bs, zp, dtype):
    c = make_case(M, N, K, bits, bs, np.float16, has_zp=zp, has_bias=True, seed=K + M)
    dev = lambda x: None if x is None else torch.from_numpy(x).cuda()
    scales = dev(c.scales).to(dtype)
    op = MatMulNBits(K, N, bits, bs, dtype=dtype, has_zero_points=zp, has_bias=True)
    assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
    if dtype == torch.float16:
        assert _lib.load().MnbGemmKernelName(M, N, K, bits, bs, _lib.DTYPE_FLOAT16).startswith(b"mnb_mid") or M <= 16
    wide = torch.full((M * (K + 24),), float("nan"), dtype=dtype, device="cuda")
    a = wide[: (M - 1) * (K + 24) + K].as_strided((M, K), (K + 24, 1))
    a.copy_(dev(c.A))
    bias = dev(c.bias).to(dtype)
    y = op.Compute(a, bias=bias).double().cpu().numpy()
    w = oracle.C.dequantize(c.B, scales.float().cpu().numpy(), c.zero_points, N, K, bits, bs).astype(np.float64)
    want = a.double().cpu().numpy() @ w.T + bias.double().cpu().numpy()
    assert np.linalg.norm(y - want) <= 5e-3 * np.linalg.norm(want)
