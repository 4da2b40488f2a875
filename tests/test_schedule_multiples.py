"""The default schedule's level-0 chains fill the device's 256 CUs in whole rounds from n = 48
on (host only): a few chains more than a multiple of 256 would run by themselves.  Lengths
differ by at most one and stay within half of the length from which more rounds are taken."""
import pytest

from chain_emulator import plan_levels


@pytest.mark.parametrize("N", [1280, 1281, 1700, 2047, 2048, 2049, 3000, 4095, 4097, 5000, 6144,
                               6500, 8192, 8193, 9000, 12288, 20000, 40000])
@pytest.mark.parametrize("n", [48, 64, 96, 128])
def test_multiples_of_the_cus(N, n):
    _, levels = plan_levels(N, n)
    lens = [c[1] for c in levels[0][1]]
    assert len(lens) % 256 == 0
    assert max(lens) - min(lens) <= 1
    assert max(lens) <= 3 * (16 if n <= 64 else 32) // 2
    if len(lens) > 256:  # fewer rounds would have had longer chains
        assert min(lens) >= (16 if n <= 64 else 32) * 2 // 3 - 1


@pytest.mark.parametrize("N", [1280, 1700, 2303, 3000, 8192])
@pytest.mark.parametrize("n", [16, 32])
def test_small_blocks(N, n):
    _, levels = plan_levels(N, n)
    lens = [c[1] for c in levels[0][1]]
    assert len(lens) == 256 if N < 2304 else len(lens) > 256
    assert max(lens) <= 9 and min(lens) >= 4
