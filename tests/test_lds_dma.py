"""The hand-written LDS-DMA loads (csrc/ek_lds_dma.h) in the device assembly
that the build's own flags give. The compiler's hazard pass does not look into
inline assembly, so what it would have seen to is checked here, on the CPU."""

import os
import re
import subprocess

import pytest

from enginekernel_amd import build as B

SOURCES = [f for f in sorted(os.listdir(B.CSRC)) if f.endswith(".hip")
           and '"ek_lds_dma.h"' in open(os.path.join(B.CSRC, f)).read()]


@pytest.fixture(scope="module", params=SOURCES)
def kernels(request, tmp_path_factory):
    """{kernel: [(opcode, instruction), ...]}; labels are ("label", name), the
    start of an inline assembly block ("label", "inline")."""
    if not os.path.exists(B.HIPCC):
        pytest.skip("needs hipcc")
    out = tmp_path_factory.mktemp("asm") / "k.s"
    r = subprocess.run([B.HIPCC, *B.FLAGS, "-S", "--cuda-device-only", os.path.join(B.CSRC, request.param),
                        "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    found, code = {}, []
    for line in out.read_text().splitlines():
        text = line.split(";")[0].strip()
        name = re.match(r"(_Z\w+):$", text)
        if name:
            code = found.setdefault(name[1], [])
        elif "#ASMSTART" in line:
            code.append(("label", "inline"))
        elif text.endswith(":"):
            code.append(("label", text))
        elif text and not text.startswith("."):
            code.append((text.split()[0], text))
    found = {k: v for k, v in found.items() if any(op.startswith("global_load_lds") for op, _ in v)}
    assert found
    return found


def _sgprs(operand):
    """The scalar registers that an operand names."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]|s(\d+)", operand)
    if not m:
        return set()
    return set(range(int(m[1]), int(m[2]) + 1)) if m[1] else {int(m[3])}


def test_wait_states_before_lds_dma(kernels):
    """A load may read m0 from one wait state after its scalar write on, and a
    scalar base from five after a vector instruction's write of it; nothing
    else uses m0."""
    for name, code in kernels.items():
        for i, (op, text) in enumerate(code):
            if not op.startswith("global_load_lds"):
                assert not re.search(r"\bm0\b", text) or op == "s_mov_b32", (name, text)
                continue
            assert "m0" not in code[i - 1][1], (name, code[i - 1][1], text)
            base = set().union(*(_sgprs(t.strip(", ")) for t in text.split()[1:]))
            waited = 0
            for prev, ptext in reversed(code[:i]):
                if prev.startswith("v_") and waited < 5:
                    assert not base & _sgprs(ptext.split()[1].strip(",")), (name, ptext, text)
                waited += 0 if prev == "label" else int(ptext.split()[1]) + 1 if prev == "s_nop" else 1
                if waited >= 5:
                    break


def test_one_wave_buffer_hand_over(kernels):
    """A workgroup of one wave has no barrier between its reads of a buffer and
    the loads that refill it: its own wait names both counters."""
    for name, code in kernels.items():
        if any(op == "s_barrier" for op, _ in code):
            continue
        waits = [text for (_, prev), (op, text) in zip(code, code[1:]) if prev == "inline" and op == "s_waitcnt"]
        assert waits and all("vmcnt(0)" in w and "lgkmcnt(0)" in w for w in waits), (name, waits)
