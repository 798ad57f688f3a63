"""The column-pair quantiser (mnb_quantize_pairs_kernel) reads the 32 rows of a wavefront by dwords with the row in a scalar offset
wherever the rows begin at multiples of four bytes, also where K or N leave a remainder.  No GPU needed."""
import re
import shutil
import subprocess

import pytest

from onnxruntime_amd import build

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    out = tmp_path_factory.mktemp("isa") / "quant.s"
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", str(build.CSRC / "mnb_quant.hip"), "-o", str(out)], check=True,
                   capture_output=True, timeout=900)
    return {m.groups(): b for b in re.split(r"^(?=_Z\w+:)", out.read_text(), flags=re.M)
            for m in [re.match(r"_ZN\S*mnb_quantize_pairs_kernelILi(\d)ELi(\d)EL\S*?(\d)EEEv\w*:", b)] if m}


def test_rows_are_read_with_their_offset_in_a_scalar_register(kernels):
    assert {k[2] for k in kernels} == {"0", "1", "2"}  # any address; multiples of four; multiples of four and no remainders
    for key, text in kernels.items():
        if key[2] == "0":
            continue
        loads = re.findall(r"^\s*buffer_load_dword v\d+, v\d+, s\[\d+:\d+\], s\d+ offen", text, re.M)
        # (the first row's offset is the constant 0)
        assert len(loads) >= 31, (key, len(loads))
