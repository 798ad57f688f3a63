"""The gather of activations by a group index, rows through LDS (mnb_variant_gather_rows_kernel): against the product with the
columns put in order by torch, bit for bit, at rows of every length modulo a load and a thread's share."""
import numpy as np
import pytest
import torch

from onnxruntime_amd import MatMulNBits
from onnxruntime_amd.synthetic import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K", [32, 36, 4096, 4100, 8232, 16384, 16420, 32768, 32800])
def test_rows_of_every_length(dtype, K):
    N, bs = 16, 32
    if K > 8232:
        N = 1
    c = make_case(1, N, K, 4, bs, np.float16, has_zp=True, seed=K)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    g_idx = torch.from_numpy(np.random.default_rng(K).permutation(K) // bs).to(torch.int32)
    op = MatMulNBits(K, N, 4, bs, dtype=dtype, has_zero_points=True, has_g_idx=True)
    assert op.PrePack(dev(c.B), dev(c.scales).to(dtype), dev(c.zero_points), g_idx.cuda())
    # unit rows read single weights back: W[:, k], exactly (float16 and float32), whatever the kernel's order of sums
    ks = [0, 1, K // 2, K - 9 if K > 9 else 2, K - 1] * 4  # (20 rows: long ones are gathered so from 17 on, in shares up to 64)
    a = torch.zeros(len(ks) + 1, K + 8, dtype=dtype, device="cuda")
    for i, k in enumerate(ks):
        a[i, k] = 1
    blob = torch.from_numpy(c.B.reshape(N, -1))
    q = torch.stack((blob & 15, blob >> 4), -1).reshape(N, -1)[:, :K].double()
    zp = torch.from_numpy(c.zero_points)
    zp = torch.stack((zp & 15, zp >> 4), -1).reshape(N, -1).double()
    scales = dev(c.scales).to(dtype).cpu().double()
    want = torch.stack([(q[:, k] - zp[:, g_idx[k]]) * scales.reshape(N, -1)[:, g_idx[k]] for k in ks]).to(dtype)
    pad = torch.zeros(len(ks), K + 1, dtype=dtype, device="cuda")
    pad[:, :K] = a[:len(ks), :K]
    for rows in (a[:len(ks), :K].contiguous(), a[:len(ks), :K], pad[:, :K]):  # pitches that 16-byte loads can read and one that they cannot
        assert torch.equal(op.Compute(rows).cpu(), want)
        assert torch.equal(op.Compute(rows[2:3]).cpu(), want[2:3])
    many = op.Compute(a[:len(ks), :K].repeat(4, 1))
    assert torch.equal(many.cpu(), want.repeat(4, 1))
    # half a million elements and more are gathered through LDS: all of the above, one row less, and pitches as above
    least = -(-(1 << 19) // K)
    times = -(-least // len(ks))
    for rows in (a[:len(ks), :K].contiguous(), a[:len(ks), :K], pad[:, :K]):
        whole = torch.empty(times * len(ks), rows.stride(0), dtype=dtype, device="cuda")[:, :K]
        whole.copy_(rows.repeat(times, 1))
        for M in (least, least - 1):
            assert torch.equal(op.Compute(whole[:M]).cpu(), want.repeat(times, 1)[:M])
