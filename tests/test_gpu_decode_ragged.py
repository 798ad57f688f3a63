"""Decode (up to 16 rows) with K beyond whole chunks of 128 (8-bit: 64) and with rows at any 16-bit address: the wavefront that takes
the rest, every weight format and type, slabs of every width, few and many chunks."""
import numpy as np
import pytest
import torch

from onnxruntime_amd import MatMulNBits, MatMulNBitsMlp, MatMulNBitsQkv, _lib
from onnxruntime_amd.synthetic import make_case
from oracle import oracle

pytestmark = pytest.mark.gpu


def dev(x):
    return None if x is None else torch.from_numpy(np.ascontiguousarray(x)).cuda()


def weights(c, scales, bits, bs):
    return oracle.C.dequantize(c.B, scales.float().cpu().numpy(), c.zero_points, c.N, c.K, bits, bs).astype(np.float64)


@pytest.mark.parametrize("bits,bs,zp,dtype", [(4, 16, True, torch.float16), (4, 32, False, torch.float16), (4, 128, True, torch.float16),
                                              (4, 256, False, torch.float16), (8, 32, True, torch.float16), (8, 128, False, torch.float16),
                                              (2, 64, True, torch.float16), (4, 32, True, torch.bfloat16), (4, 128, True, torch.bfloat16),
                                              (4, 256, False, torch.bfloat16), (8, 64, True, torch.bfloat16), (2, 128, False, torch.bfloat16)])
# one column; slabs of one, two, (three,) and four tiles; K of one value to one less than a chunk beyond 1, 15, 16, 33 and 65 chunks
@pytest.mark.parametrize("N,K", [(1, 129), (37, 255), (300, 2047), (5136, 1921), (9000, 328), (12900, 260), (40, 4227), (500, 8392)])
def test_products(N, K, bits, bs, zp, dtype):
    c = make_case(16, N, K, bits, bs, np.float16, has_zp=zp, has_bias=True, seed=N + K)
    op = MatMulNBits(K, N, bits, bs, dtype=dtype, has_zero_points=zp, has_bias=True)
    scales, bias = dev(c.scales).to(dtype), dev(c.bias).to(dtype)
    assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
    # NaN around every row: what stands behind K must not count.  Rows at every address modulo 16 bytes.
    pitch = K + 5
    store = torch.full((17 * pitch + 8,), float("nan"), dtype=dtype, device="cuda")
    # rounding of each weight and of the result to the 16-bit type: 2^-11 (bfloat16 2^-8) each, relative
    tol = 2e-3 if dtype == torch.float16 else 1e-2
    w = weights(c, scales, bits, bs)
    for M, first in ((1, 0), (3, 1), (4, 0), (8, 6), (16, 3)):
        a = store[first:first + M * pitch].view(M, pitch)[:, :K]
        a.copy_(dev(c.A[:M]))
        want = a.double().cpu().numpy() @ w.T + bias.double().cpu().numpy()
        y = op.Compute(a, bias=bias)
        assert np.linalg.norm(y.double().cpu().numpy() - want) <= tol * np.linalg.norm(want), (M, first)
        store.fill_(float("nan"))


@pytest.mark.parametrize("M", [1, 7])
@pytest.mark.parametrize("bits,bs,K", [(4, 32, 712), (8, 64, 328), (4, 128, 1400), (4, 32, 264)])
def test_fused_outputs(M, bits, bs, K):
    g, u, q, k, v = (make_case(M, n, K, bits, bs, np.float16, has_bias=True, seed=s) for s, n in enumerate((90, 90, 91, 37, 37)))
    a = dev(g.A)
    alone = lambda c: a.double().cpu().numpy() @ weights(c, dev(c.scales), bits, bs).T + c.bias.astype(np.float64)  # noqa: E731
    parts = lambda c: (dev(c.B), dev(c.scales), dev(c.bias))  # noqa: E731
    close = lambda got, want: np.linalg.norm(got.double().cpu().numpy() - want) <= 3e-3 * np.linalg.norm(want)  # noqa: E731
    mlp, qkv = MatMulNBitsMlp(K, 90, bits, bs), MatMulNBitsQkv(K, 91, 37, bits, bs)
    assert mlp.PrePack(*parts(g), *parts(u)) and qkv.PrePack(*parts(q), *parts(k), *parts(v))
    gf, uf = alone(g), alone(u)
    assert close(mlp.Compute(a), gf / (1 + np.exp(-gf)) * uf)
    for got, c in zip(qkv.Compute(a), (q, k, v)):
        assert close(got, alone(c))


def test_without_scratch_and_the_names():
    lib = _lib.load()
    assert lib.MnbGemmKernelName(1, 4096, 4104, 4, 64, _lib.DTYPE_FLOAT16) == b"mnb_skinny_kernel"
    assert lib.MnbGemmKernelName(16, 4096, 100, 4, 64, _lib.DTYPE_FLOAT16).startswith(b"mnb_mid")
    c = make_case(5, 70, 200, 4, 32, np.float16, seed=3)
    op = MatMulNBits(200, 70, 4, 32)
    assert op.PrePack(dev(c.B), dev(c.scales))
    a, y = dev(c.A), torch.empty(5, 70, dtype=torch.float16, device="cuda")
    _lib.check(lib.MnbGemm(5, 70, 200, 4, 32, 0, _lib.DTYPE_FLOAT16, a.data_ptr(), 200, op.packed.data_ptr(), None, y.data_ptr(), 70,
                           None, 0, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(y, op.Compute(a))


@pytest.mark.parametrize("bits,bs,zp,dtype", [(4, 128, True, torch.float16), (4, 256, False, torch.float16), (8, 64, True, torch.float16),
                                              (8, 128, False, torch.float16), (2, 128, True, torch.float16), (4, 32, True, torch.float16),
                                              (4, 128, True, torch.bfloat16), (4, 256, False, torch.bfloat16)])
# slabs of one, two and four tiles; one chunk, several turns; what stands beyond them
@pytest.mark.parametrize("N,K", [(37, 255), (300, 2047), (5136, 520), (12900, 392)])
def test_infinities_stay_infinities(N, K, bits, bs, zp, dtype):
    """An infinite activation makes each column infinite whose weight is not zero, of the weight's sign; a NaN makes all of them NaN."""
    c = make_case(16, N, K, bits, bs, np.float16, has_zp=zp, has_bias=True, seed=N + K)
    op = MatMulNBits(K, N, bits, bs, dtype=dtype, has_zero_points=zp, has_bias=True)
    scales, bias = dev(c.scales).to(dtype), dev(c.bias).to(dtype)
    assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
    w = weights(c, scales, bits, bs)
    inf = float("inf")
    for M in (1, 3, 6, 16):
        for k in (0, K // 2, K - 1):
            a = dev(c.A[:M]).to(dtype)
            a[M - 1, k] = inf
            if M > 1:
                a[0, K - 1 - k // 2] = -inf
            if M > 4:
                a[2, k], a[3, k], a[3, k - 1] = float("nan"), inf, -inf
            with np.errstate(invalid="ignore"):
                want = a.double().cpu().numpy() @ w.T + bias.double().cpu().numpy()
            got = op.Compute(a, bias=bias).double().cpu().numpy()
            same = np.isfinite(want)
            assert np.array_equal(np.isfinite(got), same) and np.array_equal(got[~same], want[~same], equal_nan=True), (M, k)
            tol = 2e-3 if dtype == torch.float16 else 1e-2  # (as above)
            assert np.linalg.norm(got[same] - want[same]) <= tol * np.linalg.norm(want[same]) + 1e-30, (M, k)


@pytest.mark.parametrize("bs,zp", [(32, True), (128, True), (256, False)])
def test_large_bfloat16_values(bs, zp):
    """Activations whose products with raw weights (128 and more) have no fp32 value, while those with the weights themselves do."""
    N, K = 300, 520
    c = make_case(4, N, K, 4, bs, np.float16, has_zp=zp, seed=8)
    op = MatMulNBits(K, N, 4, bs, dtype=torch.bfloat16, has_zero_points=zp)
    scales = dev(c.scales).to(torch.bfloat16)
    assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
    a = (dev(c.A).float() * 1e36).to(torch.bfloat16)
    want = a.double().cpu().numpy() @ weights(c, scales, 4, bs).T
    got = op.Compute(a).double().cpu().numpy()
    assert np.linalg.norm(got - want) <= 1e-2 * np.linalg.norm(want)  # (as above)


# 4-bit, odd pitches: beside the widths (12784, 16384, 24576) and the rows (5, 9) where tiles, wavefronts and the way through LDS change; fewer
# chunks than wavefronts, one turn of them and one step, several turns
@pytest.mark.parametrize("bs,zp,dtype", [(32, True, torch.float16), (128, False, torch.float16), (64, False, torch.bfloat16),
                                         (128, True, torch.bfloat16)])
@pytest.mark.parametrize("N,K,rows", [(12785, 391, (1, 4, 5, 16)), (16384, 4233, (4, 9, 16)), (16385, 2049, (4, 8, 9)), (24577, 1029, (4, 5, 16)),
                                      (8193, 2184, (8, 9, 16))])
def test_wide_matrices_rows_between_words(N, K, rows, bs, zp, dtype):
    c = make_case(16, N, K, 4, bs, np.float16, has_zp=zp, seed=N + K)
    op = MatMulNBits(K, N, 4, bs, dtype=dtype, has_zero_points=zp)
    scales, a = dev(c.scales).to(dtype), dev(c.A).to(dtype)
    assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
    want = a.double().cpu().numpy() @ weights(c, scales, 4, bs).T
    tol = 2e-3 if dtype == torch.float16 else 1e-2  # (as above)
    for M in rows:
        y = op.Compute(a[:M])
        assert np.linalg.norm(y.double().cpu().numpy() - want[:M]) <= tol * np.linalg.norm(want[:M]), M


# the streaming kernel's side of the line and the decode kernel's: chunks (128, 8-bit 64) before the rest, what the rest lacks, columns
@pytest.mark.parametrize("bits,N,K,short", [(4, 37, 136, True), (4, 16, 136, False), (4, 17, 264, True), (4, 300, 488, True), (4, 300, 496, False), (4, 64, 520, False), (4, 64, 300, False),
                                            (4, 4096, 264, True), (4, 4097, 264, False), (8, 50, 232, True), (8, 50, 248, True),
                                            (8, 50, 264, False), (2, 40, 392, True)])
def test_short_k(bits, N, K, short):
    assert (_lib.load().MnbGemmKernelNameStrided(9, N, K, bits, 32, _lib.DTYPE_FLOAT16, K) == b"mnb_mid_kernel") == short
    c = make_case(16, N, K, bits, 32, np.float16, has_zp=True, seed=N + K)
    op = MatMulNBits(K, N, bits, 32, has_zero_points=True)
    assert op.PrePack(dev(c.B), dev(c.scales), dev(c.zero_points))
    a = torch.full((16, K + 8), float("nan"), dtype=torch.float16, device="cuda")
    a[:, :K] = dev(c.A)
    want = c.A.astype(np.float64) @ weights(c, dev(c.scales), bits, 32).T
    for M in (1, 9, 16):
        for pitch in (K, K + 8):
            rows = a[:M, :K] if pitch > K else dev(c.A[:M])
            y, without = op.Compute(rows), torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
            assert np.linalg.norm(y.double().cpu().numpy() - want[:M]) <= 2e-3 * np.linalg.norm(want[:M]), M  # (as above)
            _lib.check(_lib.load().MnbGemm(M, N, K, bits, 32, 1, _lib.DTYPE_FLOAT16, rows.data_ptr(), pitch, op.packed.data_ptr(), None,
                                           without.data_ptr(), N, None, 0, torch.cuda.current_stream().cuda_stream))
            assert torch.equal(without, y), M  # (the scratch that such calls bring decides nothing)
