"""Partition counts (host rule of the library, no GPU)."""
import pytest

from blockgtq_amd import _capi


@pytest.mark.parametrize("rule", ["bgtq_default_splits", "bgtq_ragged_splits"])
def test_counts_stay_in_range_and_never_start_a_round_for_a_remainder(rule):
    pick = getattr(_capi.lib(), rule)
    for pairs in [1, 2, 3, 7, 8, 16, 24, 48, 100, 128, 129, 160, 255, 256, 257, 700, 4096, 2**20]:
        for T in [1, 64, 127, 128, 129, 3001, 8192, 131072, 2**31 - 1]:
            n = pick(1, pairs, T)
            assert 1 <= n <= min(512, -(-T // 128))
            if 1 < n < min(512, -(-T // 128)):      # one more partition would have cost another round
                assert -(-pairs * (n + 1) // 256) > -(-pairs * n // 256)
    assert pick(0, 8, 100) == pick(1, 0, 100) == pick(1, 8, 0) == 1


def test_counts_of_measured_shapes():
    lib = _capi.lib()
    assert [lib.bgtq_default_splits(*s) for s in [(8, 2, 32768), (1, 8, 131072), (4, 2, 8200), (12, 4, 3001), (20, 8, 8192)]] == [16, 32, 32, 5, 3]
    assert [lib.bgtq_ragged_splits(*s) for s in [(12, 4, 3001), (8, 2, 32768), (16, 4, 8192), (4, 8, 16384), (32, 8, 4096), (32, 8, 16384)]] == [5, 16, 4, 8, 1, 4]
