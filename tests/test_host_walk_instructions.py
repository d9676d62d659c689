"""The instructions of the forward's walk, from the assembly of ``fwd.hip`` as it is built: around the matrix
instructions of the kernel that long launches run, nothing computes LDS addresses (they are constants plus
one register each), and nothing is spilled."""
import os
import re
import subprocess

import pytest

from ultraattn_amd.build import CSRC, HIPCC_FLAGS, hipcc_path


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "fwd.s"
    cmd = [hipcc_path(), *HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, "fwd.hip"), "-o", str(out)]
    try:
        r = subprocess.run(cmd, capture_output=True, text=True)
    except FileNotFoundError:
        pytest.skip("no hipcc")
    assert r.returncode == 0, r.stderr
    return out.read_text()


def _blocks(text, kernel):
    """Basic blocks (lists of instructions) of one kernel."""
    body = re.search(rf"^{kernel}\w*:.*?^\.Lfunc_end", text, flags=re.M | re.S).group(0)
    blocks = re.split(r"^(?:\.LBB\w+:|; %bb\.\d+:).*$", body, flags=re.M)
    return [re.findall(r"^[ \t]+((?:[vs]|ds|buffer)_\w+)[ \t]*(.*)$", b, flags=re.M) for b in blocks]


def test_no_address_arithmetic_between_matrix_instructions(assembly):
    walk = [b for b in _blocks(assembly, "_ZN2ua10fwd_kernelILi1E") if any("mfma" in op for op, _ in b)]
    assert sum("mfma" in op for b in walk for op, _ in b) >= 64              # two half tiles, two products of 16 each
    integer = [f"{op} {args}" for b in walk for op, args in b if re.match(r"v_\w*(?:_u32|_i32|_b32|_u64|_b64)", op)]
    assert not integer, integer


def test_nothing_spilled(assembly):
    spills = re.findall(r"\.vgpr_spill_count:\s*(\d+)", assembly)
    assert spills and all(s == "0" for s in spills)
