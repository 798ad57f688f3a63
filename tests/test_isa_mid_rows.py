"""The waits of the streaming kernel's many-row form (mnb_mid_rows.hip.h) count the vector-memory operations that are younger
than what they wait for.  That holds as long as the generated code issues exactly the operations that the source counts (a
load that nothing uses would be dropped): for every instantiation the operations of the assembly are walked through, two turns
of the loop and the tail, with and without the loop.  No GPU needed."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from onnxruntime_amd import build

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
STAGES = 4


@pytest.fixture(scope="module")
def blocks(tmp_path_factory):
    out = tmp_path_factory.mktemp("isa") / "mid.s"
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"] + build.EXTRA_FLAGS.get("mnb_mid.hip", [])
    subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", str(build.CSRC / "mnb_mid.hip"), "-o", str(out)], check=True,
                   capture_output=True, timeout=900)
    found = {}
    for block in re.split(r"^(?=_Z\w+:)", out.read_text(), flags=re.M):
        m = re.match(r"_ZN\S*mnb_mid_shared_rows_kernelILi(\d)ELb(\d)ELi(\d)ELi(\d)ELi(\d)E\w*:", block)
        if m:
            found[m.groups()] = block
    return found


@pytest.fixture(scope="module")
def kernels(blocks):
    return {key: block[:block.index("s_endpgm")] for key, block in blocks.items()}


def events(text):
    """('dma' | 'load' | ('wait', n) | 'barrier') of a piece of the listing, in order."""
    got = []
    for line in text.split("\n"):
        t = line.split(";")[0].strip()
        if re.match(r"buffer_load\S* .* lds$", t):
            got.append("dma")
        elif re.match(r"(buffer|global)_(load|store|atomic)", t):
            got.append("load")
        elif t.startswith("s_waitcnt") and "vmcnt" in t:
            got.append(("wait", int(re.search(r"vmcnt\((\d+)\)", t).group(1))))
        elif t.startswith("s_barrier"):
            got.append("barrier")
    return got


def walk(trace, rt, what):
    """Every barrier finds the chunk's rt fill instructions complete."""
    issued, fills, done, chunk = 0, [], 0, 0
    for e in trace:
        if e in ("dma", "load"):
            if e == "dma":
                fills.append(issued)
            issued += 1
        elif e == "barrier":
            assert len(fills) >= (chunk + 1) * rt, f"{what}: chunk {chunk} has not been asked for"
            assert fills[(chunk + 1) * rt - 1] < done, f"{what}: chunk {chunk} may be in flight behind its barrier"
            chunk += 1
        else:
            done = max(done, issued - e[1])
    return chunk


def test_every_barrier_finds_its_chunk_in_lds(kernels):
    assert len(kernels) == 8 * (2 + 2 + 1 + 2 + 2)  # tiles x (4-bit fp16, bfloat16, typed zero points; 8-bit fp16, bfloat16)
    for key, text in kernels.items():
        rt = int(key[2])
        header = re.search(r"^(\.LBB\d+_\d+):.*Loop Header", text, re.M)
        label = header.group(1)
        back = [m for m in re.finditer(r"s_cbranch_\w+ " + re.escape(label) + r"\b", text) if m.start() > header.start()]
        head, body, rest = text[:header.start()], text[header.start():back[-1].end()], text[back[-1].end():]
        head, body, rest = events(head), events(body), events(rest)
        assert body.count("barrier") == STAGES and body.count("dma") == STAGES * rt, key
        # the tail: up to three chunks, which ask for nothing; behind it everything is waited for
        end, seen = 0, 0
        while seen < 3:
            seen += rest[end] == "barrier"
            end += 1
        tail = rest[:end]
        assert "dma" not in tail and "load" not in tail, key
        assert walk(head + body + body + tail, rt, key) == 2 * STAGES + 3
        assert walk(head + tail, rt, key) == 3
        assert ("wait", 0) in rest[end:end + rest[end:].index("barrier")], key


def test_a_compute_unit_holds_the_workgroups_that_the_estimate_of_the_tiles_assumes(blocks):
    """Two wavefronts a SIMD for every workgroup of eight, 32 KB of LDS for every row tile."""
    for key, block in blocks.items():
        bits, _, rt, cw, _ = map(int, key)
        assumed = {1: 2 if bits == 8 and cw == 4 else 4, 2: 2, 3: 1, 4: 1}[rt]  # (mid_rows_per_cu)
        wavefronts = int(re.search(r"; Occupancy: (\d+)", block).group(1))
        held = min(wavefronts // 2, 160 // (32 * rt))
        assert held == assumed if rt == 1 else held >= assumed, (key, wavefronts)
        assert re.search(r"; ScratchSize: 0\b", block), key
