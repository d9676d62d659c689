"""The benchmark's probes exist and check their arguments before they launch anything: every loop whose rate bench.py counts as a ceiling."""
import pytest

import bench


@pytest.mark.parametrize("rows,reuse,turn", bench.MFMA_REUSE)
def test_mfma_loops_with_operands_used_again(rows, reuse, turn):
    lib, host = bench.probe_lib(), 16                                            # an address that is never read
    assert lib.bench_probe_mfma_reuse(None, None, 1, 1, rows, reuse, turn, None) == -1
    assert lib.bench_probe_mfma_reuse(host, host, 0, 1, rows, reuse, turn, None) == -2
    assert lib.bench_probe_mfma_reuse(host, host, 1, 1, rows + 1, reuse, turn, None) == -2
    assert lib.bench_probe_mfma_reuse(host, host, 1, 1, rows, 3, turn, None) == -2
    assert lib.bench_probe_mfma_reuse(host + 4, host, 1, 1, rows, reuse, turn, None) == -4
    assert bench.mfma_reuse_key(rows, reuse, turn).startswith("random_")         # (what `measured_ceiling_tflops` takes)


def test_what_the_ceiling_covers():
    """Either instruction with operands that change every time and with an A operand used twice, as the walks use theirs."""
    assert {(16, 1, 0), (16, 2, 0), (32, 1, 0), (32, 2, 0)} <= set(bench.MFMA_REUSE)
