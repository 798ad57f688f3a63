"""One row of MatMulNBitsMlp / MatMulNBitsQkv with the normalisation inside the projection (mnb_skinny_norm.hip), against
the separate normalisation followed by the same operator without one.

The two add the squares of the row in different orders (relative difference of the sum at most 2 K 2^-24, mostly far less),
so the normalised halves are equal or neighbours (relative 2^-10), and by Cauchy-Schwarz a result of the product moves by at
most 2^-10 |a| |w|; the results are narrowed to fp16 once more (2^-10 relative for both together).  The MLP adds silu'(g) <= 1.1
and a product of the two factors: gated on the relative L2 instead, 4 2^-10."""
import numpy as np
import pytest
import torch

from onnxruntime_amd import _lib
from onnxruntime_amd.matmul_nbits import MatMulNBitsMlp, MatMulNBitsQkv

pytestmark = pytest.mark.gpu


def weights(rng, n, k, bits, bs):
    kb = k // bs if k % bs == 0 else k // bs + 1
    b = torch.from_numpy(rng.integers(0, 256, size=(n, kb, bs * bits // 8), dtype=np.uint8)).cuda()
    s = torch.from_numpy(rng.uniform(0.001, 0.01, size=(n, kb)).astype(np.float16)).cuda()
    return b, s, None


def half(rng, *shape):
    return torch.from_numpy(rng.standard_normal(shape).astype(np.float16)).cuda()


def separate(op, a, norm, skip):
    """The normalised row and A + skip in the operators' own arithmetic: fp32 sums, narrowed once."""
    x = a.float() + (skip.float() if skip is not None else 0)
    denom = torch.sqrt((x * x).mean(dim=-1, keepdim=True) + op.epsilon)
    return (x / denom * norm.float()).half(), x.half()


# K: fewer chunks than wavefronts, one to several per wavefront with every remainder, the longest row; columns: single-,
# two- and four-tile slabs, ragged
@pytest.mark.parametrize("K", [128, 640, 1152, 2944, 4096, 4224, 8192])
@pytest.mark.parametrize("Nq,Nkv", [(48, 16), (500, 37), (4096, 1024), (8000, 2500)])
@pytest.mark.parametrize("bits,bs", [(4, 32), (4, 128), (4, 16), (8, 64), (8, 32)])
def test_qkv(K, Nq, Nkv, bits, bs):
    rng = np.random.default_rng(K + Nq + bs)
    op = MatMulNBitsQkv(K, Nq, Nkv, bits, bs)
    assert op.PrePack(*weights(rng, Nq, K, bits, bs), *weights(rng, Nkv, K, bits, bs), *weights(rng, Nkv, K, bits, bs))
    a, norm, skip = half(rng, 1, K), 1 + half(rng, K) * 0.1, half(rng, 1, K)
    for sk in (None, skip):
        got = op.Compute(a, norm_scale=norm, skip=sk, want_skip_sum=sk is not None)
        row, total = separate(op, a, norm, sk)
        want = op.Compute(row)
        if sk is not None:
            assert torch.equal(got[3], total)
        for g, w in zip(got[:3], want[:3]):
            g, w = g.double(), w.double()
            assert torch.linalg.norm(g - w) <= 2**-9 * torch.linalg.norm(w)


@pytest.mark.parametrize("K,N", [(128, 16), (1152, 1000), (4096, 14336), (8192, 520)])
@pytest.mark.parametrize("bits,bs", [(4, 32), (4, 128), (8, 64)])
def test_mlp(K, N, bits, bs):
    rng = np.random.default_rng(K + N + bs)
    op = MatMulNBitsMlp(K, N, bits, bs)
    assert op.PrePack(*weights(rng, N, K, bits, bs), *weights(rng, N, K, bits, bs))
    a, norm, skip = half(rng, 1, K), 1 + half(rng, K) * 0.1, half(rng, 1, K)
    got, total = op.Compute(a, skip=skip, norm_scale=norm, want_skip_sum=True)
    row, want_total = separate(op, a, norm, skip)
    want = op.Compute(row)
    assert torch.equal(total, want_total)
    assert torch.linalg.norm(got.double() - want.double()) <= 2**-8 * torch.linalg.norm(want.double())


def test_outputs_on_the_inputs():
    """A sum written over the skip row (or Q over A) reads its inputs first: the separate normalisation runs."""
    rng = np.random.default_rng(1)
    K, Nq, Nkv = 4096, 4096, 1024
    op = MatMulNBitsQkv(K, Nq, Nkv, 4, 128)
    assert op.PrePack(*weights(rng, Nq, K, 4, 128), *weights(rng, Nkv, K, 4, 128), *weights(rng, Nkv, K, 4, 128))
    a, norm, skip = half(rng, 1, K), 1 + half(rng, K) * 0.1, half(rng, 1, K)
    want = op.Compute(a, norm_scale=norm, skip=skip, want_skip_sum=True)
    lib, F16 = _lib.load(), _lib.DTYPE_FLOAT16
    need = lib.MnbQkvWorkspaceSize(1, Nq, Nkv, K, 4, 128, F16, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    k, v = torch.empty_like(want[1]), torch.empty_like(want[2])
    n = _lib.MnbNormPrologue()
    n.norm_scale_dev, n.skip_dev, n.ld_skip, n.epsilon = norm.data_ptr(), skip.data_ptr(), K, op.epsilon
    n.skip_sum_dev, n.ld_skip_sum = skip.data_ptr(), K
    import ctypes
    _lib.check(lib.MnbQkvGemm(1, Nq, Nkv, K, 4, 128, F16, a.data_ptr(), K, ctypes.byref(n), op.packed.data_ptr(),
                              a.data_ptr(), Nq, k.data_ptr(), Nkv, v.data_ptr(), Nkv, ws.data_ptr(), need,
                              torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(skip, want[3])
    for g, w in ((a, want[0]), (k, want[1]), (v, want[2])):
        assert torch.linalg.norm(g.double() - w.double()) <= 2**-9 * torch.linalg.norm(w.double())
