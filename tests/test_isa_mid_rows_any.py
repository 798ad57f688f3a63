"""The same checks of the generated code for the many-row form's kernels with a ragged last chunk or a cut along K
(mnb_mid_any.hip), whose first loads are others."""
import re
import subprocess

import pytest

from isa_hazard_scan import scan
from onnxruntime_amd import build
from tests import test_isa_mid_rows as checks


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    out = tmp_path_factory.mktemp("isa") / "mid_any.s"
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"] + build.EXTRA_FLAGS["mnb_mid_any.hip"]
    subprocess.run([checks.HIPCC, *flags, "--cuda-device-only", "-S", str(build.CSRC / "mnb_mid_any.hip"), "-o", str(out)],
                   check=True, capture_output=True, timeout=900)
    return out.read_text()


@pytest.fixture(scope="module")
def blocks(listing):
    found = {}
    for block in re.split(r"^(?=_Z\w+:)", listing, flags=re.M):
        m = re.match(r"_ZN\S*mnb_mid_shared_rows_kernelILi(\d)ELb(\d)ELi(\d)ELi(\d)ELi(\d)ELb1E\w*:", block)
        if m:
            found[m.groups()] = block
    return found


def test_no_early_read_of_mfma_results(listing):
    findings = scan(listing)
    assert not findings, "\n".join(f"{f}: {w} wait states: {a} -> {b}" for f, w, a, b in findings[:10])


kernels = checks.kernels
for _name in [n for n in dir(checks) if n.startswith("test_")]:
    globals()[_name] = getattr(checks, _name)
