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
