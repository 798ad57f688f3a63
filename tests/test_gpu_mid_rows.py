"""The streaming kernel's many-row form (mnb_mid_rows.hip.h): every tile, chunk counts around its four stages, ragged rows and
columns, all types.  The tile is forced through the calibration library's override; the product's own choice is
timed against others in test_gpu_plans.py and named in test_host_logic.py."""
import ctypes
import os

import numpy as np
import pytest
import torch

from onnxruntime_amd import MatMulNBits, MatMulNBitsMlp, MatMulNBitsQkv, _lib
from onnxruntime_amd.calibration import build as cal_build
from onnxruntime_amd.synthetic import make_case
from oracle import oracle

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not cal_build.lib_path().exists(),
                                                  reason="the calibration library has not been built")]
TILES = [(rt, cw) for cw in (2, 4) for rt in (1, 2, 3, 4)]


@pytest.fixture
def forced(monkeypatch):
    product, cal = _lib.load(), ctypes.CDLL(str(cal_build.lib_path()))
    for name in ("MnbGemm", "MnbVariantGemm", "MnbGemmWorkspaceSize", "MnbVariantGemmWorkspaceSize", "MnbMlpGemm",
                 "MnbMlpWorkspaceSize", "MnbQkvGemm", "MnbQkvWorkspaceSize", "MnbGetLastErrorMessage"):
        getattr(cal, name).restype, getattr(cal, name).argtypes = getattr(product, name).restype, getattr(product, name).argtypes
    monkeypatch.setenv("MNB_MID_MAX_M", "99999")

    def use(op, rt, cw):
        monkeypatch.setenv("MNB_MID_ROWS", f"{rt},{cw}")
        op.lib = _Mixed(cal, product)
        return op
    yield use


class _Mixed:
    """Products of the calibration library, everything else (packing) of the product's."""

    def __init__(self, cal, product):
        self.cal, self.product = cal, product

    def __getattr__(self, name):
        return getattr(self.cal if name.endswith(("Gemm", "WorkspaceSize")) else self.product, name)


def dev(x):
    return None if x is None else torch.from_numpy(np.ascontiguousarray(x)).cuda()


@pytest.mark.parametrize("rt,cw", TILES)
@pytest.mark.parametrize("bits,bs,zp,dtype", [(4, 32, True, torch.float16), (4, 128, False, torch.float16),
                                              (4, 256, True, torch.float16), (8, 32, True, torch.float16),
                                              (8, 64, False, torch.float16), (2, 64, True, torch.float16),
                                              (4, 64, True, torch.bfloat16), (4, 32, False, torch.bfloat16),
                                              (8, 32, True, torch.bfloat16), (8, 256, False, torch.bfloat16)])
def test_tiles(forced, rt, cw, bits, bs, zp, dtype):
    # chunks of 128: one, around the four stages, several turns of them; rows and columns off the tile, one tile and several
    for (M, N, chunks) in ((17, 33, 1), (64, 300, 2), (97, 130, 3), (129, 65, 4), (130, 1000, 5), (33, 520, 7), (250, 257, 18)):
        K = 128 * chunks
        c = make_case(M, N, K, bits, bs, np.float16, has_zp=zp, has_bias=True, seed=M + chunks)
        op = MatMulNBits(K, N, bits, bs, dtype=dtype, has_zero_points=zp, has_bias=True)
        scales = dev(c.scales).to(dtype)
        assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
        store = torch.full((M, K + 24), float("nan"), dtype=dtype, device="cuda")  # NaN behind every row
        a = store[:, :K]
        a.copy_(dev(c.A))
        bias = dev(c.bias).to(dtype)
        y = forced(op, rt, cw).Compute(a, bias=bias)
        w = oracle.C.dequantize(c.B, scales.float().cpu().numpy(), c.zero_points, N, K, bits, bs).astype(np.float64)
        want = a.double().cpu().numpy() @ w.T + bias.double().cpu().numpy()
        got = y.double().cpu().numpy()
        # rounding of each weight and of the result to the 16-bit type: 2^-11 (bfloat16 2^-8) each, relative
        tol = 2e-3 if dtype == torch.float16 else 1e-2
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want), (M, N, K)
        assert torch.equal(op.Compute(a, bias=bias), y)


@pytest.mark.parametrize("rt,cw", TILES)
@pytest.mark.parametrize("M,N,K", [(300, 4100, 1408), (1211, 2488, 1664)])
def test_many_workgroups_give_the_same_bits_as_other_tiles_give_sums(forced, rt, cw, M, N, K):
    """More workgroups than the chip holds, chunk counts of 3 modulo 4: unit-vector rows return columns of W bit for bit."""
    c = make_case(M, N, K, 4, 32, np.float16, has_zp=True, seed=1)
    ks = np.random.default_rng(0).integers(0, K, size=M)
    eye = np.zeros((M, K), np.float16)
    eye[np.arange(M), ks] = 1
    op = MatMulNBits(K, N, 4, 32, has_zero_points=True)
    assert op.PrePack(dev(c.B), dev(c.scales), dev(c.zero_points))
    w = oracle.C.dequantize(c.B, c.scales, c.zero_points, N, K, 4, 32)
    want = np.ascontiguousarray(w[:, ks].T).view(np.uint16)
    for _ in range(3):
        y = forced(op, rt, cw).Compute(dev(eye)).cpu().numpy()
        assert np.array_equal(y.view(np.uint16), want)


@pytest.mark.parametrize("rt,cw", TILES)
@pytest.mark.parametrize("K,bits,bs", [(640, 4, 32), (648, 4, 32), (1400, 4, 256), (120, 8, 64), (904, 8, 128)])
def test_fused_outputs(forced, rt, cw, K, bits, bs):
    """gate / up and Q, K, V of odd widths: the same values as the separate products of the same library.  Whole chunks of 128, and a last
    one that is not whole."""
    M = 70
    mats = [make_case(M, n, K, bits, bs, np.float16, has_bias=True, seed=n) for n in (90, 91, 37, 53)]
    a = dev(mats[0].A)

    def alone(c):
        w = oracle.C.dequantize(c.B, c.scales, None, c.N, K, bits, bs).astype(np.float64)
        return a.double().cpu().numpy() @ w.T + c.bias.astype(np.float64)
    parts = lambda c: (dev(c.B), dev(c.scales), dev(c.bias))  # noqa: E731
    close = lambda got, want: np.linalg.norm(got.double().cpu().numpy() - want) <= 3e-3 * np.linalg.norm(want)  # noqa: E731
    g, u = (make_case(M, 90, K, bits, bs, np.float16, has_bias=True, seed=s) for s in (1, 2))
    mlp = MatMulNBitsMlp(K, 90, bits, bs)
    assert mlp.PrePack(*parts(g), *parts(u))
    gf, uf = alone(g), alone(u)
    assert close(forced(mlp, rt, cw).Compute(a), gf / (1 + np.exp(-gf)) * uf)
    qkv = MatMulNBitsQkv(K, 91, 37, bits, bs)
    k, v = mats[2], make_case(M, 37, K, bits, bs, np.float16, has_bias=True, seed=9)
    assert qkv.PrePack(*parts(mats[1]), *parts(k), *parts(v))
    for got, c in zip(forced(qkv, rt, cw).Compute(a), (mats[1], k, v)):
        assert got.shape[1] == c.N and close(got, alone(c))


@pytest.mark.parametrize("rt,cw", TILES)
@pytest.mark.parametrize("K", [256, 264])
def test_rows_behind_the_result_are_not_stored(forced, rt, cw, K):
    """Tiles that end in and behind the last row, and those of 96 rows, whose threads store in steps of 64: the 48 rows behind the
    result keep what they hold."""
    for M, N in ((17, 130), (65, 64), (96, 257), (97, 128), (192, 90), (200, 256)):
        c = make_case(M, N, K, 4, 32, np.float16, seed=M)
        op = MatMulNBits(K, N, 4, 32)
        assert op.PrePack(dev(c.B), dev(c.scales))
        store = torch.full((M + 48, N), float("nan"), dtype=torch.float16, device="cuda")
        forced(op, rt, cw).Compute(dev(c.A), out=store[:M])
        w = oracle.C.dequantize(c.B, c.scales, None, N, K, 4, 32).astype(np.float64)
        want = c.A.astype(np.float64) @ w.T
        assert np.linalg.norm(store[:M].double().cpu().numpy() - want) <= 2e-3 * np.linalg.norm(want), (M, N)  # (as above)
        assert torch.isnan(store[M:]).all(), (M, N)


@pytest.mark.parametrize("rt,cw", [(1, 2), (2, 4), (4, 4)])
@pytest.mark.parametrize("bits,bs,zp,dtype", [(4, 32, True, torch.float16), (4, 256, False, torch.float16),
                                              (8, 64, True, torch.float16), (4, 64, True, torch.bfloat16)])
def test_rows_that_only_a_padded_copy_serves(forced, rt, cw, bits, bs, zp, dtype):
    """A ragged K, an odd pitch, an odd address; whole chunks with rows that 16-byte loads must not read."""
    for (M, N, K, pitch, first) in ((17, 130, 130, 130, 0), (65, 300, 249, 256, 0), (70, 90, 1275, 1275, 1), (129, 257, 1000, 1008, 8),
                                    (40, 260, 384, 385, 0), (33, 64, 512, 520, 3)):
        c = make_case(M, N, K, bits, bs, np.float16, has_zp=zp, seed=M + K)
        op = MatMulNBits(K, N, bits, bs, dtype=dtype, has_zero_points=zp)
        scales = dev(c.scales).to(dtype)
        assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
        store = torch.full((M * pitch + first,), float("nan"), dtype=dtype, device="cuda")  # NaN around every row
        a = store[first:].view(M, pitch)[:, :K]
        a.copy_(dev(c.A))
        y = forced(op, rt, cw).Compute(a)
        w = oracle.C.dequantize(c.B, scales.float().cpu().numpy(), c.zero_points, N, K, bits, bs).astype(np.float64)
        want = a.double().cpu().numpy() @ w.T
        tol = 2e-3 if dtype == torch.float16 else 1e-2  # (as above)
        assert np.linalg.norm(y.double().cpu().numpy() - want) <= tol * np.linalg.norm(want), (M, N, K)


@pytest.mark.parametrize("rt,cw", TILES)
@pytest.mark.parametrize("bits,bs,zp,dtype", [(4, 32, True, torch.float16), (4, 128, False, torch.float16),
                                              (4, 256, True, torch.float16), (8, 32, True, torch.float16),
                                              (8, 256, False, torch.float16), (2, 64, True, torch.float16),
                                              (4, 256, True, torch.bfloat16), (8, 64, True, torch.bfloat16)])
def test_a_ragged_last_chunk_is_read_in_place(forced, rt, cw, bits, bs, zp, dtype):
    """K a multiple of 8: one chunk that is not whole, around the four stages and several turns of them.  What stands behind K, in the
    rows' padding, behind the matrix and in LDS from the launch before, is no number and must not count."""
    for (M, N, K, pitch) in ((17, 33, 8, 8), (64, 300, 120, 136), (97, 130, 136, 136), (33, 65, 320, 328), (130, 520, 504, 1024),
                             (65, 257, 520, 520), (70, 129, 760, 768), (250, 140, 2248, 2256)):
        c = make_case(M, N, K, bits, bs, np.float16, has_zp=zp, has_bias=True, seed=M + K)
        op = MatMulNBits(K, N, bits, bs, dtype=dtype, has_zero_points=zp, has_bias=True)
        scales = dev(c.scales).to(dtype)
        assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
        store = torch.full((M + 2, pitch), float("nan"), dtype=dtype, device="cuda")
        a = store[:M, :K]
        a.copy_(dev(c.A))
        bias = dev(c.bias).to(dtype)
        forced(op, rt, cw)
        assert torch.isnan(op.Compute(torch.full((600, K), float("nan"), dtype=dtype, device="cuda"))).all()
        y = op.Compute(a, bias=bias)
        w = oracle.C.dequantize(c.B, scales.float().cpu().numpy(), c.zero_points, N, K, bits, bs).astype(np.float64)
        want = a.double().cpu().numpy() @ w.T + bias.double().cpu().numpy()
        tol = 2e-3 if dtype == torch.float16 else 1e-2  # (as above)
        assert np.linalg.norm(y.double().cpu().numpy() - want) <= tol * np.linalg.norm(want), (M, N, K)


@pytest.mark.parametrize("rt,cw", TILES)
@pytest.mark.parametrize("bits,bs,zp,dtype", [(4, 32, True, torch.float16), (4, 256, False, torch.float16), (8, 256, True, torch.float16),
                                              (2, 64, True, torch.float16), (4, 256, True, torch.bfloat16), (8, 32, False, torch.bfloat16)])
def test_k_cut_over_workgroups(forced, monkeypatch, rt, cw, bits, bs, zp, dtype):
    """Cuts of equal and unequal chunks, the last one of a single chunk and of one that is not whole; the scratch holds NaN before."""
    for (M, N, K, cuts) in ((17, 33, 1024, 2), (65, 90, 1160, 3), (130, 129, 2176, 4), (97, 65, 2320, 8), (33, 40, 4088, 5), (250, 70, 3336, 7)):
        c = make_case(M, N, K, bits, bs, np.float16, has_zp=zp, has_bias=True, seed=M + K)
        op = MatMulNBits(K, N, bits, bs, dtype=dtype, has_zero_points=zp, has_bias=True)
        scales = dev(c.scales).to(dtype)
        assert op.PrePack(dev(c.B), scales, dev(c.zero_points))
        a = torch.full((M, K + 8), float("nan"), dtype=dtype, device="cuda")[:, :K]
        a.copy_(dev(c.A))
        bias = dev(c.bias).to(dtype)
        forced(op, rt, cw)
        whole = op.Compute(a, bias=bias)
        monkeypatch.setenv("MNB_MID_ROWS", f"{rt},{cw},{cuts}")
        assert op._workspace
        for ws in op._workspace.values():
            ws.fill_(255)
        y = op.Compute(a, bias=bias)
        assert all((ws != 255).any() for ws in op._workspace.values()), (M, N, K, cuts)  # the sums of the cuts
        w = oracle.C.dequantize(c.B, scales.float().cpu().numpy(), c.zero_points, N, K, bits, bs).astype(np.float64)
        want = a.double().cpu().numpy() @ w.T + bias.double().cpu().numpy()
        tol = 2e-3 if dtype == torch.float16 else 1e-2  # (as above)
        err = lambda t: np.linalg.norm(t.double().cpu().numpy() - want) / np.linalg.norm(want)  # noqa: E731
        # the same products in another order of fp32 sums: no further from 64 bits than uncut, but for single roundings of the result
        assert err(y) <= tol and err(y) <= 1.1 * err(whole) + 1e-6, (M, N, K, cuts)
        assert torch.equal(y, op.Compute(a, bias=bias))


def test_the_planner_cuts_narrow_matrices_of_long_k():
    M, N, K = 168, 745, 7680
    c = make_case(M, N, K, 4, 64, np.float16, has_zp=True, seed=2)
    op = MatMulNBits(K, N, 4, 64, has_zero_points=True)
    assert op.PrePack(dev(c.B), dev(c.scales), dev(c.zero_points))
    a = dev(c.A)
    op.Compute(a)
    for ws in op._workspace.values():
        ws.fill_(255)
    y = op.Compute(a)
    assert any((ws != 255).any() for ws in op._workspace.values())  # the sums of the cuts
    w = oracle.C.dequantize(c.B, c.scales, c.zero_points, N, K, 4, 64).astype(np.float64)
    want = a.double().cpu().numpy() @ w.T
    assert np.linalg.norm(y.double().cpu().numpy() - want) <= 2e-3 * np.linalg.norm(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        z = op.Compute(a)
    for _ in range(3):
        z.zero_()
        op.Compute(a)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, y)


@pytest.mark.parametrize("M,N,K,bs", [(2186, 1833, 50048, 128), (573, 7206, 51200, 64)])
def test_scratch_beyond_what_a_call_asks_for_is_not_used(M, N, K, bs):
    """Sizes of the tile GEMM that the many-row form takes over ask for no scratch: with some they give the same bits, and leave it alone."""
    lib, f16, stream = _lib.load(), _lib.DTYPE_FLOAT16, torch.cuda.current_stream().cuda_stream
    assert lib.MnbGemmWorkspaceSize(M, N, K, 4, bs, 0, f16) == 0
    assert lib.MnbGemmKernelName(M, N, K, 4, bs, f16) == b"mnb_mid_shared_rows_kernel"
    make = torch.Generator(device="cuda").manual_seed(1)
    op = MatMulNBits(K, N, 4, bs)
    assert op.PrePack(torch.randint(0, 256, (N, K // bs, bs // 2), generator=make, device="cuda", dtype=torch.uint8),
                      torch.rand(N, K // bs, generator=make, device="cuda").half() * 0.01)
    a = torch.randn(M, K, generator=make, device="cuda").half()
    much = torch.full((256 << 20,), 255, dtype=torch.uint8, device="cuda")
    y = [torch.empty(M, N, dtype=torch.float16, device="cuda") for _ in range(2)]
    for out, ws, size in ((y[0], None, 0), (y[1], much.data_ptr(), much.numel())):
        _lib.check(lib.MnbGemm(M, N, K, 4, bs, 0, f16, a.data_ptr(), K, op.packed.data_ptr(), None, out.data_ptr(), N, ws, size, stream))
    assert torch.equal(*y) and bool((much == 255).all())
