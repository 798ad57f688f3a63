"""The planners' choices against the alternatives they could have made, timed on the device.

Needs the calibration library (python -m onnxruntime_amd.calibration.build: the product sources with the planners'
environment overrides compiled in); skipped when it has not been built.  For each problem the plan the library picks
by itself must be within 25 % of the fastest forced alternative (HIP graphs of 20 launches, best of three): a plan
that is off by more than box-to-box noise fails here instead of going unnoticed."""
import ctypes
import os

import numpy as np
import pytest
import torch

from onnxruntime_amd import _lib
from onnxruntime_amd.calibration import build as cal_build
from onnxruntime_amd.calibration import run as cal_run
from onnxruntime_amd.matmul_nbits import MatMulNBitsMlp, MatMulNBitsQkv, quantize_blockwise, simplified_layer_norm

pytestmark = pytest.mark.gpu

CAL = cal_build.lib_path()


def _time(call, launches=20, reps=3):
    best = float("inf")
    for _ in range(reps):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(launches):
                assert call() == 0
        g.replay()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        g.replay()
        g.replay()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) / (2 * launches) * 1e3)
    return best


# (M, N, K, bits, block, copies of the packed matrix), alternatives as environment settings
CASES = [
    ((1, 14336, 4096, 4, 128, 16), ["MNB_SKINNY_PLAN=4,8", "MNB_SKINNY_PLAN=2,16", "MNB_SKINNY_PLAN=2,8"]),
    ((1, 6144, 4096, 4, 64, 16), ["MNB_SKINNY_PLAN=4,16", "MNB_SKINNY_PLAN=1,16", "MNB_SKINNY_PLAN=2,8"]),
    ((1, 14336, 4096, 2, 128, 16), ["MNB_SKINNY_PLAN=4,8", "MNB_SKINNY_PLAN=2,16", "MNB_SKINNY_MODE=1"]),
    # few rows on single-tile slabs (activations through LDS or read straight from A), long K on four-tile slabs
    # (eight wavefronts with the straight-line loop or sixteen with conditional prefetches), the gate+up decode plan
    ((4, 4096, 14336, 4, 128, 32), ["MNB_SKINNY_A4=0", "MNB_SKINNY_PLAN=2,8", "MNB_SKINNY_PLAN=1,16"]),
    ((16, 14336, 8192, 4, 128, 16), ["MNB_SKINNY_T4LDS=0", "MNB_SKINNY_PLAN=2,8"]),
    ((1, 28672, 4096, 4, 128, 16), ["MNB_SKINNY_PLAN=4,8", "MNB_SKINNY_PLAN=2,8", "MNB_SKINNY_PLAN=2,4"]),
    # the streaming kernels: many rows on tiles that all wavefronts share, pairs of wavefronts that share activations (with the
    # first switched off), tiles of 16 columns; the tile GEMM
    ((64, 28672, 4096, 4, 128, 1), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=0,0+MNB_MID_SHARED=0", "MNB_MID_ROWS=2,2", "MNB_MID_ROWS=1,4"]),
    ((64, 28672, 4096, 8, 64, 8), ["MNB_MID_SHARED=0", "MNB_MID_ROWS=2,4", "MNB_MID_ROWS=2,2"]),
    ((64, 20000, 2048, 8, 64, 16), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=1,4", "MNB_MID_ROWS=2,2"]),
    ((64, 4096, 14336, 4, 128, 1), ["MNB_MID_PLAN=1,4,8", "MNB_MID_PLAN=2,2,4", "MNB_MID_SHARED=1", "MNB_MID_ROWS=2,2"]),
    ((256, 6144, 4096, 4, 128, 1), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=4,2", "MNB_MID_ROWS=2,4", "MNB_MID_MAX_M=64+MNB_MID_ROWS=0,0"]),
    ((128, 11008, 4096, 4, 128, 16), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=2,4", "MNB_MID_ROWS=4,2", "MNB_MID_ROWS=3,4"]),
    ((681, 2113, 512, 8, 128, 24), ["MNB_MID_ROWS=0,0+MNB_MID_MAX_M=64", "MNB_MID_ROWS=1,2+MNB_MID_MAX_M=9999", "MNB_MID_ROWS=2,4+MNB_MID_MAX_M=9999"]),
    ((1024, 4096, 4096, 4, 128, 16), ["MNB_MID_MAX_M=64", "MNB_MID_ROWS=4,2+MNB_MID_MAX_M=9999", "MNB_MID_ROWS=3,4+MNB_MID_MAX_M=9999"]),
    ((2111, 1881, 6144, 8, 128, 16), ["MNB_MID_MAX_M=64", "MNB_MID_ROWS=4,2+MNB_MID_MAX_M=9999"]),
    ((1225, 10845, 1152, 4, 128, 16), ["MNB_MID_MAX_M=64", "MNB_MID_ROWS=4,4+MNB_MID_MAX_M=9999"]),
    # many rows of long K, few columns: activations that go through the fabric once per slab
    ((3543, 333, 13056, 4, 32, 4), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=3,2+MNB_MID_MAX_M=9999", "MNB_MID_ROWS=2,4+MNB_MID_MAX_M=9999"]),
    ((6915, 241, 5632, 8, 32, 4), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=4,2+MNB_MID_MAX_M=9999", "MNB_MID_ROWS=2,4+MNB_MID_MAX_M=9999"]),
    ((2242, 2008, 7360, 4, 64, 8), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=3,2"]),
    # ragged K: the same from a padded copy, or the forms that need none
    ((1366, 2378, 4056, 4, 32, 16), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=2,2"]),
    ((138, 12513, 272, 4, 32, 24), ["MNB_MID_ROWS=0,0", "MNB_MID_ROWS=1,4"]),
    ((45, 534, 5411, 4, 32, 24), ["MNB_MID_ROWS=1,2"]),
    # ragged K: activations in place or from the staged copy
    ((31, 4778, 7400, 8, 64, 16), ["MNB_MID_DIRECT=0"]),
    ((59, 2633, 11976, 8, 64, 16), ["MNB_MID_DIRECT=0"]),
    ((48, 5940, 3640, 4, 32, 24), ["MNB_MID_DIRECT=0"]),
    ((37, 5003, 2880, 4, 32, 24), ["MNB_MID_DIRECT=0"]),
    ((18, 1452, 3544, 8, 64, 24), ["MNB_MID_DIRECT=0"]),
    ((1024, 4096, 14336, 4, 128, 1), ["MNB_GEMM256_PLAN=256,1", "MNB_GEMM256_PLAN=128,2", "MNB_MID_MAX_M=4096"]),
    ((2048, 14336, 4096, 4, 32, 1), ["MNB_GEMM256_PLAN=128,1", "MNB_GEMM256_WAVES=4"]),
]


@pytest.mark.skipif(not CAL.exists(), reason="the calibration library has not been built")
@pytest.mark.parametrize("shape,alternatives", CASES)
def test_the_plan_chosen_is_close_to_the_best_alternative(shape, alternatives):
    M, N, K, bits, bs, copies = shape
    lib = cal_run.load(str(CAL))
    prob = cal_run.Problem(M, N, K, bits, bs, zp=True, bias=False, copies=copies)
    times = {}
    try:
        for env in [""] + alternatives:
            cal_run.set_env(dict(kv.split("=", 1) for kv in env.split("+") if kv))
            call, _ = prob.caller(lib)
            print("plan", env or "(chosen)", shape, flush=True)   # (names the case should a launch fault)
            assert call() == 0
            torch.cuda.synchronize()
            for _ in range(50):   # clock and caches settled
                call()
            torch.cuda.synchronize()
            times[env] = _time(call, launches=max(20, copies))
    finally:
        cal_run.set_env({})
    chosen, best = times[""], min(times.values())
    # (one alternative that differs in the activations' way alone, nothing else: closer)
    limit = 1.1 if alternatives == ["MNB_MID_DIRECT=0"] else 1.25
    assert chosen <= limit * best, f"{shape}: chosen {chosen:.1f} us, alternatives {times}"


# [K, N] fp16, tiles in runs along K or strips side by side: rows that 16-byte loads cannot read and rows that they can, few tiles
# and many, every width
@pytest.mark.skipif(not CAL.exists(), reason="the calibration library has not been built")
@pytest.mark.parametrize("K,N,bits,bs,zp", [(4096, 130, 2, 32, True), (8192, 33, 2, 32, True), (4096, 1001, 4, 32, True),
                                            (4096, 4095, 2, 128, True), (4096, 4095, 4, 32, False), (4832, 12825, 4, 32, False),
                                            (4096, 14336, 8, 128, False), (4096, 14336, 4, 128, False), (4096, 14336, 4, 64, True),
                                            (4096, 14336, 4, 16, False), (4096, 14336, 4, 256, False)])
def test_the_order_of_the_quantisers_tiles_is_close_to_the_other(K, N, bits, bs, zp):
    lib, product = ctypes.CDLL(str(CAL)), _lib.load()
    lib.MnbQuantizeBlockwise.restype = product.MnbQuantizeBlockwise.restype
    lib.MnbQuantizeBlockwise.argtypes = product.MnbQuantizeBlockwise.argtypes
    sources = [torch.randn(K, N, device="cuda").half() for _ in range(max(1, min(48, (1 << 29) // (2 * K * N))))]  # from HBM
    turn = iter(range(10**9))
    b = torch.empty(N, -(-K // bs), bs * bits // 8, dtype=torch.uint8, device="cuda")
    s = torch.empty(N, -(-K // bs), dtype=torch.float16, device="cuda")
    z = torch.empty(N, (-(-K // bs) * bits + 7) // 8, dtype=torch.uint8, device="cuda") if zp else None

    def call():
        return lib.MnbQuantizeBlockwise(b.data_ptr(), s.data_ptr(), None if z is None else z.data_ptr(),
                                        sources[next(turn) % len(sources)].data_ptr(), bs, bits, K, N, N, _lib.DTYPE_FLOAT16,
                                        torch.cuda.current_stream().cuda_stream)

    times = {}
    try:
        for env in ("", "MNB_QUANT_RUNS=0", "MNB_QUANT_RUNS=1"):
            cal_run.set_env(dict(kv.split("=", 1) for kv in env.split("+") if kv))
            for _ in range(50):
                assert call() == 0
            torch.cuda.synchronize()
            times[env] = _time(call, launches=48, reps=5)
    finally:
        cal_run.set_env({})
    assert times[""] <= 1.1 * min(times.values()), times


# a last block that K cuts short is no reason to take longer than for a whole one: small matrices, where a workgroup's own time
# shows, and ordinary ones
@pytest.mark.parametrize("K,N,bits,bs,zp,dtype", [(200, 13, 4, 32, False, torch.float16), (1105, 71, 8, 32, True, torch.float16),
                                                  (600, 1001, 2, 64, False, torch.float16), (288, 4756, 4, 128, False, torch.float16),
                                                  (1083, 3924, 8, 128, False, torch.float16), (600, 1001, 4, 32, False, torch.float32),
                                                  (288, 4756, 4, 128, False, torch.float32), (300, 128, 4, 256, True, torch.float32)])
def test_the_quantiser_takes_no_longer_for_a_ragged_last_block(K, N, bits, bs, zp, dtype):
    times = []
    rows = 4 * bs if bs <= 64 else bs  # (short blocks go up to four to a workgroup)
    for k in (K, -(-K // rows) * rows):
        sources = [torch.randn(k, N, device="cuda").to(dtype) for _ in range(24)]
        turn = iter(range(10**9))

        def call():
            quantize_blockwise(sources[next(turn) % 24], bits, bs, not zp)
            return 0
        for _ in range(50):
            call()
        torch.cuda.synchronize()
        times.append(_time(call, launches=24, reps=5))
    # (0.2 us for the rows that are filled in; measured before the last block went the way of the others: 1.2 to 1.9 times)
    assert times[0] <= 1.1 * times[1] + 0.2, times


# fp32 prefill on the bfloat16 matrix cores or on the fp32 ones: short K in several turns of workgroups, ordinary prompts
@pytest.mark.skipif(not CAL.exists(), reason="the calibration library has not been built")
@pytest.mark.parametrize("M,N,K,bits,bs", [(293, 9315, 256, 8, 128), (1052, 1928, 256, 4, 16), (544, 9786, 128, 8, 16),
                                           (1345, 4168, 128, 4, 16), (512, 4096, 4096, 4, 32), (130, 4096, 1024, 4, 32),
                                           (300, 1000, 512, 4, 32), (45, 6036, 2858, 4, 128), (27, 8554, 972, 4, 32),
                                           (196, 1327, 3615, 4, 128), (44, 5673, 3087, 8, 64), (52, 2805, 794, 8, 64), (51, 7554, 980, 4, 64),
                                           (73, 6412, 668, 4, 64), (518, 589, 962, 4, 64), (47, 18892, 23, 4, 32)])
def test_the_fp32_kernel_chosen_is_close_to_the_other(M, N, K, bits, bs):
    lib, product = ctypes.CDLL(str(CAL)), _lib.load()
    for name in ("MnbGemm", "MnbGemmWorkspaceSize"):
        getattr(lib, name).restype = getattr(product, name).restype
        getattr(lib, name).argtypes = getattr(product, name).argtypes
    size = product.MnbPackQuantBDataSize(N, K, bits, bs, 1, _lib.DTYPE_FLOAT)
    packed = torch.full((size,), 0x1c, dtype=torch.uint8, device="cuda")   # (small scales and zero points, whatever they are)
    a, y = torch.randn(M, K, device="cuda"), torch.empty(M, N, device="cuda")
    times = {}
    try:
        for env in ("", "MNB_GEMM32_SPLIT=0", "MNB_GEMM32_SPLIT=y"):
            cal_run.set_env(dict(kv.split("=", 1) for kv in env.split("+") if kv))
            need = lib.MnbGemmWorkspaceSize(M, N, K, bits, bs, 1, _lib.DTYPE_FLOAT)
            ws = torch.empty(need + 1, dtype=torch.uint8, device="cuda")

            def call():
                return lib.MnbGemm(M, N, K, bits, bs, 1, _lib.DTYPE_FLOAT, a.data_ptr(), K, packed.data_ptr(), None,
                                   y.data_ptr(), N, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
            for _ in range(50):
                assert call() == 0
            torch.cuda.synchronize()
            times[env] = _time(call, reps=5)
    finally:
        cal_run.set_env({})
    assert times[""] <= 1.1 * min(times.values()), times


# (K, columns of Q and of K and V, or of the MLP), bits, block: three-tile slabs, raw two-tile slabs beyond 512 tiles, one to
# 1.6 rounds and one round of four-tile slabs, where the decode kernel's own plan is the better one; and single-, two- and
# four-tile slabs where the normalisation belongs inside
@pytest.mark.parametrize("K,n,bits,bs", [(8192, (3072, 3072), 4, 128), (2048, (5504,), 4, 128), (8192, (16384, 2048), 4, 32),
                                         (8192, (8192,), 4, 32), (4096, (2048, 512), 4, 128), (4096, (4096, 1024), 4, 128),
                                         (4096, (14336,), 4, 128)])
def test_one_row_with_its_normalisation_is_no_slower_than_the_two_steps(K, n, bits, bs):
    """MatMulNBitsMlp / MatMulNBitsQkv of one row against the normalisation and the plain operator one after the other."""
    g = torch.Generator(device="cuda").manual_seed(K)

    def weights(cols):
        b = torch.randint(0, 256, (cols, K // bs, bs * bits // 8), generator=g, device="cuda", dtype=torch.uint8)
        return b, torch.rand(cols, K // bs, generator=g, device="cuda").mul(0.01).half(), None

    def make():
        op = MatMulNBitsMlp(K, n[0], bits, bs) if len(n) == 1 else MatMulNBitsQkv(K, *n, bits, bs)
        cols = [n[0], n[0]] if len(n) == 1 else [n[0], n[1], n[1]]
        assert op.PrePack(*[t for c in cols for t in weights(c)])
        return op

    ops = [make() for _ in range(8)]
    a, skip = (torch.randn(1, K, generator=g, device="cuda").half() for _ in range(2))
    scale = torch.ones(K, device="cuda", dtype=torch.float16)
    turn = iter(range(10**9))

    def together():
        ops[next(turn) % 8].Compute(a, skip=skip, norm_scale=scale, want_skip_sum=True)
        return 0

    def apart():
        op = ops[next(turn) % 8]
        op.Compute(simplified_layer_norm(a, scale, op.epsilon, skip, want_skip_sum=True)[0])
        return 0

    times = {}
    for call in (together, apart):
        for _ in range(50):
            call()
        torch.cuda.synchronize()
        times[call] = _time(call, launches=24, reps=5)
    assert times[together] <= 1.1 * times[apart], f"together {times[together]:.2f} us, apart {times[apart]:.2f} us"
