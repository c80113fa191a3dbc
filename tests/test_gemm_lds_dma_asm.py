"""Wait states the hardware asks of the program in front of the transforms'
global -> LDS loads, which are issued as inline assembly (fribo_gemm.hip), so
that the compiler inserts none: one between a scalar write of M0, which holds
the LDS address, and the load; five between a vector instruction's write of a
scalar register and a load that reads it (CDNA3 ISA, "Manually Inserted Wait
States").  Also, no LDS read of a wave may be outstanding when it passes the
workgroup barrier after which the next loads overwrite the stage it read."""
import os
import re
import shutil
import subprocess

import pytest

from fribois2d_amd import build


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    hipcc = build.HIPCC
    if not (os.path.exists(hipcc) or shutil.which(hipcc)):
        pytest.skip("no hipcc")
    out = str(tmp_path_factory.mktemp("asm") / "gemm.s")
    flags = [f for f in build.FLAGS if f not in ("-shared", "-fPIC")]
    subprocess.run([hipcc, *flags, "--offload-device-only", "-S", os.path.join(build.CSRC, "fribo_gemm.hip"), "-o",
                    out], check=True, capture_output=True)
    found, cur = {}, None
    with open(out) as f:
        for line in f:
            s = line.split(";")[0].strip()
            m = re.match(r"(_Z\w*gemm_dma\w*):$", s)
            if m:
                cur = found.setdefault(m.group(1), [])
            elif s.startswith(".Lfunc_end"):
                cur = None
            elif cur is not None and s and not (s.startswith(".") and not s.endswith(":")):
                cur.append(s)
    assert len(found) >= 10
    return found


def _states(ins):
    m = re.match(r"s_nop (\w+)", ins)
    return int(m.group(1), 0) + 1 if m else 1


def _sregs(text):
    """Scalar registers named in an operand list."""
    regs = set()
    for m in re.finditer(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        regs.update(range(int(m.group(1)), int(m.group(2)) + 1) if m.group(1) else [int(m.group(3))])
    return regs


def test_wait_states_before_the_lds_loads(kernels):
    seen = 0
    for name, code in kernels.items():
        for i, ins in enumerate(code):
            if not ins.startswith("global_load_lds"):
                continue
            seen += 1
            base = _sregs(ins)
            states = 0
            for prev in reversed(code[max(0, i - 8):i]):
                if re.match(r"s_\w+ m0\b", prev):
                    assert states >= 1, (name, prev, ins)
                if prev.startswith("v_") and states < 5:
                    assert not (_sregs(prev.split(",")[0]) & base), (name, prev, ins)
                states += 0 if prev.endswith(":") else _states(prev)
    assert seen >= 60


def test_no_lds_read_outstanding_at_a_barrier(kernels):
    for name, code in kernels.items():
        pending = False
        for ins in code:
            if ins.startswith("ds_read"):
                pending = True
            elif re.match(r"s_waitcnt .*lgkmcnt\(0\)", ins):
                pending = False
            elif ins == "s_barrier":
                assert not pending, name
