"""The instructions of the walks, from the assembly of ``fwd.hip`` and ``bwd.hip`` as they are built: around the matrix
instructions of the forward that long launches run, nothing computes LDS addresses (they are constants plus
one register each), and what long launches run spills nothing."""
import os
import re
import subprocess

import pytest

from ultraattn_amd.build import CSRC, HIPCC_FLAGS, hipcc_path


def _assemble(tmp_path_factory, source):
    out = tmp_path_factory.mktemp("asm") / (source + ".s")
    cmd = [hipcc_path(), *HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, source), "-o", str(out)]
    try:
        r = subprocess.run(cmd, capture_output=True, text=True)
    except FileNotFoundError:
        pytest.skip("no hipcc")
    assert r.returncode == 0, r.stderr
    return out.read_text()


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    return _assemble(tmp_path_factory, "fwd.hip")


@pytest.fixture(scope="module")
def backward_assembly(tmp_path_factory):
    return _assemble(tmp_path_factory, "bwd.hip")


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


def _spills(text, what):
    """{kernel: registers spilled} of one assembly; `what` = sgpr or vgpr."""
    kernels = re.findall(r"^ +- \.agpr_count:.*?\.wavefront_size", text, flags=re.M | re.S)
    return {re.search(r"\.name:\s*(\w+)", k).group(1): int(re.search(rf"\.{what}_spill_count:\s*(\d+)", k).group(1)) for k in kernels}


def test_no_scalars_in_vector_lanes(assembly, backward_assembly):
    """One group per workgroup (form 1), what launches of more than a few hundred lines run."""
    spills = {**_spills(assembly, "sgpr"), **_spills(backward_assembly, "sgpr")}
    form_1 = {k: n for k, n in spills.items() if "kernelILi" not in k or "kernelILi1E" in k}
    assert len(form_1) == 6 and all(n <= 2 for n in form_1.values()), form_1


def test_no_vector_registers_spilled_in_the_backward(backward_assembly):
    spills = _spills(backward_assembly, "vgpr")
    assert len(spills) == 6 and not any(spills.values()), spills
