"""What the attention kernels ask of the device, from the metadata of ``fwd.hip`` and ``bwd.hip`` as they are built."""
import os
import re
import subprocess

import pytest

from ultraattn_amd.build import CSRC, HIPCC_FLAGS, hipcc_path


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """{source: assembly}"""
    out = {}
    for source in ("fwd.hip", "bwd.hip"):
        path = tmp_path_factory.mktemp("asm") / (source + ".s")
        cmd = [hipcc_path(), *HIPCC_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, source), "-o", str(path)]
        try:
            r = subprocess.run(cmd, capture_output=True, text=True)
        except FileNotFoundError:
            pytest.skip("no hipcc")
        assert r.returncode == 0, r.stderr
        out[source] = path.read_text()
    return out


def _metadata(assembly, what):
    """{kernel: value} over both sources."""
    kernels = [k for text in assembly.values() for k in re.findall(r"^ +- \.agpr_count:.*?\.wavefront_size", text, flags=re.M | re.S)]
    return {re.search(r"\.name:\s*(\w+)", k).group(1): int(re.search(rf"\.{what}:\s*(\d+)", k).group(1)) for k in kernels}


def test_no_kernel_has_a_private_segment(assembly):
    """One of 20 bytes, which no instruction used, made a backward of half lines and the launch before it longer."""
    sizes = _metadata(assembly, "private_segment_fixed_size")
    assert len(sizes) >= 12 and not any(sizes.values()), sizes


# One group of waves a workgroup: what launches of more than a few hundred lines run, and all tile lists.
ONE_GROUP = ["fwd_kernelILi1ELb0EE", "fwd_kernelILi1ELb1EE", "fwd_plain_kernelILi16EE", "fwd_short_kernelILi16EE",
             "bwd_kernelILi1ELb0EE", "bwd_kernelILi1ELb1EE", "11dkdv_kernelE", "9dq_kernelE"]
SEVERAL = ["fwd_kernelILi2ELb1EE", "fwd_kernelILi4ELb1EE", "bwd_kernelILi3ELb1EE", "bwd_kernelILi4ELb1EE"]


def test_one_group_keeps_its_registers(assembly):
    """All kernels of one group by name: no scalars in vector lanes, no vector registers in memory."""
    scalars, vectors = _metadata(assembly, "sgpr_spill_count"), _metadata(assembly, "vgpr_spill_count")
    for name in scalars:
        assert sum(n in name + "E" for n in ONE_GROUP + SEVERAL) == 1, name
    for n in ONE_GROUP:
        found = [name for name in scalars if n in name]
        assert len(found) == 1 and scalars[found[0]] == vectors[found[0]] == 0, (n, found)
    assert not any(vectors.values()), vectors


# (two half tiles, two products: 64 of 32x32x16 or 128 of 16x16x32)
@pytest.mark.parametrize("kernel,mfmas", [("fwd_kernelILi1ELb0EE", 128), ("fwd_kernelILi1ELb1EE", 64), ("fwd_plain_kernelILi16EE", 128)])
def test_no_address_arithmetic_between_matrix_instructions_of_either_kind(assembly, kernel, mfmas):
    body = re.search(rf"^_ZN2ua\d+{kernel}\w*:.*?^\.Lfunc_end", assembly["fwd.hip"], flags=re.M | re.S).group(0)
    blocks = [re.findall(r"^[ \t]+((?:[vs]|ds|buffer)_\w+)[ \t]*(.*)$", b, flags=re.M) for b in re.split(r"^(?:\.LBB\w+:|; %bb\.\d+:).*$", body, flags=re.M)]
    walk = [b for b in blocks if any("mfma" in op for op, _ in b)]
    assert sum("mfma" in op for b in walk for op, _ in b) == mfmas
    integer = [f"{op} {args}" for b in walk for op, args in b if re.match(r"v_\w*(?:_u32|_i32|_b32|_u64|_b64)", op)]
    assert not integer, integer


@pytest.mark.parametrize("kernel", ["bwd_kernelILi1ELb0EE", "bwd_kernelILi1ELb1EE", "dkdv_kernelE"])
def test_diagonal_tiles_do_not_wait_for_every_read(assembly, kernel):
    """The block of dK/dV's second products on diagonal tiles (32 MFMAs, 32 transposing reads): its waits leave the next fragment's reads in flight,
    but for the last fragment's (and the first one's at most)."""
    body = re.search(rf"^_ZN2ua\d+{kernel}\w*:.*?^\.Lfunc_end", assembly["bwd.hip"], flags=re.M | re.S).group(0)
    found = 0
    for b in re.split(r"^(?:\.LBB\w+:|; %bb\.\d+:).*$", body, flags=re.M):
        if b.count("v_mfma") == 32 and b.count("ds_read_b64_tr_b16") == 32:
            found += 1
            assert len(re.findall(r"lgkmcnt\(0\)", b)) <= 2, kernel
    assert found == 2                                       # either half of a tile


def test_rows_leave_the_forward_whole(assembly):
    """No kernel of the forward writes O in pieces of 8 bytes, 32 bytes of a row at a time: rows pass through LDS (the statistics are single dwords)."""
    stores = set(re.findall(r"^\s+(global_store_\w+)", assembly["fwd.hip"], flags=re.M))
    assert "global_store_dwordx4" in stores and stores <= {"global_store_dwordx4", "global_store_dword"}, stores


def test_short_lists_do_not_wait_for_every_read(assembly):
    """The blocks of the second products (16 MFMAs, 32 transposing reads, of which the first are in the block before or in this one): the waits leave
    reads in flight, but for the last fragment's."""
    body = re.search(r"^_ZN2ua\d+fwd_short_kernel\w*:.*?^\.Lfunc_end", assembly["fwd.hip"], flags=re.M | re.S).group(0)
    found = 0
    for b in re.split(r"^(?:\.LBB\w+:|; %bb\.\d+:).*$", body, flags=re.M):
        if b.count("v_mfma") == 16 and b.count("ds_read_b64_tr_b16") >= 16:
            found += 1
            assert len(re.findall(r"lgkmcnt\(0\)", b)) <= 2
    assert found >= 2                                       # either half of a tile


def test_accumulators_are_cleared_in_pairs(assembly):
    """No block of a one-group kernel clears 64 or 128 accumulator registers one by one."""
    for text in assembly.values():
        for body in re.findall(r"^_ZN2ua\d+\w*kernel\w*:.*?^\.Lfunc_end", text, flags=re.M | re.S):
            if any(n in body.split(":", 1)[0] + "E" for n in ONE_GROUP):
                most = max(b.count("v_mov_b32") for b in re.split(r"^(?:\.LBB\w+:|; %bb\.\d+:).*$", body, flags=re.M))
                assert most < 64, (body[:60], most)


def test_short_dense_walks_do_not_wait_for_parameters_at_their_end(assembly):
    """The dense forward of one group has nearly all it needs at its end in scalar registers (of 19 loads of parameters eight came behind the products)."""
    body = re.search(r"^_ZN2ua\d+fwd_kernelILi1ELb1EE\w*:.*?^\.Lfunc_end", assembly["fwd.hip"], flags=re.M | re.S).group(0)
    assert len(re.findall(r"s_load_dword", body[body.rindex("v_mfma"):])) <= 2


def test_no_scalars_in_vector_lanes_in_any_form(assembly):
    spilled = _metadata(assembly, "sgpr_spill_count")
    assert not any(spilled.values()), spilled
