"""The decode kernel's plan (skinny_plan in csrc/mnb_skinny_kernels.hip.h), compiled for the host.  No GPU needed."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "onnxruntime_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
PROGRAM = r"""
#include "mnb_skinny_kernels.hip.h"
const MnbDeviceInfo& mnb_device_info() { static const MnbDeviceInfo info{256, 2.4e9}; return info; }
int main() {
  int n;
  long long N, K, M;
  for (int bits, bs, zp, io; (n = scanf("%lld %lld %lld %d %d %d %d", &M, &N, &K, &bits, &bs, &zp, &io)) == 7;) {
    const MnbLayout L = mnb_make_layout(N, K, bits, bs, io == kMnbIoModel ? kMnbDtypeFloat16 : kMnbDtypeFloat, zp);
    const SkinnyPlan p = skinny_plan(L, io, M, K >= 4 * L.group_k, 1);
    printf("%d %d %d %d %zu\n", p.mode, p.t, p.nw, p.a_lds, p.smem);
  }
}
"""


def planner(d, program):
    (d / "plan.hip").write_text(program)
    subprocess.run([HIPCC, "--cuda-host-only", "-O1", "-std=c++17", "-w", "-I", str(CSRC), str(d / "plan.hip"), "-o", str(d / "plan")],
                   check=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "plan")], input=text, check=True, capture_output=True, text=True).stdout.splitlines()
        assert len(out) == len(cases)
        return [tuple(map(int, line.split())) for line in out]
    return run


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    return planner(tmp_path_factory.mktemp("skinny_plan"), PROGRAM)


@pytest.fixture(scope="module")
def plans_between_words(tmp_path_factory):
    return planner(tmp_path_factory.mktemp("skinny_plan_words"), PROGRAM.replace("L.group_k, 1)", "L.group_k, 1, false)"))


def test_ragged_k_is_planned_for_the_loop_that_runs(plans):
    """K beyond whole chunks runs the general loop whatever its chunks: on slabs of four tiles sixteen rows through LDS, from thirteen rows
    or beyond 32 chunks and nine rows on with raw 4-bit weights, or none; never the forms that load all chunks up front."""
    cases = [(M, N, K, 4 if bits == 2 else bits, bs, zp, io) for M in (1, 2, 4, 5, 8, 9, 12, 13, 16) for N in (13000, 14336, 28672)
             for K in (520, 1032, 2056, 2060, 3080, 4104, 4136, 8200, 8201) for bits, bs in ((4, 32), (4, 128), (4, 256), (8, 64), (8, 128))
             for zp in (0, 1) for io in (0, 1)]
    four = 0
    for (M, N, K, bits, bs, zp, io), (mode, t, nw, a_lds, smem) in zip(cases, plans(cases)):
        if K % (512 // bits) == 0 or t != 4:
            continue
        four += 1
        loop = bits == 4 and mode == 0 and M >= 9 and (M >= 13 or K // 128 > 32)
        assert a_lds == (16 if loop else 0) and nw in (4, 8), (M, N, K, bits, bs, zp, io)
        assert smem >= nw * t * 1024 and (not a_lds or smem >= nw * 4096)
    assert four > 500


def test_rows_between_words(plans, plans_between_words):
    """4-bit weights, K beyond whole chunks, four-tile slabs: rows of A that begin between words pass through LDS from five rows on, or the slabs
    are narrowed to two tiles (more than one round of them, up to 1.6, or three of the narrow ones a unit).  All else is planned as for rows at words."""
    cases = [(M, N, K, bits, bs, zp, io) for M in (1, 4, 5, 8, 9, 13, 16) for N in (40, 6000, 9000, 12784, 12785, 16384, 16385, 24576, 24577, 26176, 26177, 28672)
             for K in (129, 515, 2055, 2177, 4097, 4225, 4249, 9001) for bits, bs in ((4, 32), (4, 128), (8, 64)) for zp in (0, 1) for io in (0, 1)]
    narrowed = passed = 0
    for case, words, plan in zip(cases, plans(cases), plans_between_words(cases)):
        M, N, K, bits, bs, zp, io = case
        mode, t, nw, a_lds, smem = plan
        if words[1] == 4 and bits == 4 and 16384 < N <= (26176 if M <= 4 else 24576) and (M <= 8 or bs == 32):
            narrowed += 1
            assert (t, nw) == (2, 4) and a_lds == (4 if M <= 4 else 8 if M <= 8 else 16) and smem >= nw * 4096, case
        elif words[1] == 4 and bits == 4 and M >= 5:
            passed += 1
            assert (mode, t, nw, a_lds) == (*words[:3], 16) and smem >= nw * 4096, case
        else:
            assert plan == words, case
        if bits == 4 and t == 2 and M >= 9 and N > 512 * 16:
            assert nw == 4, case
    assert narrowed > 100 and passed > 100
