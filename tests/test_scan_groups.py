"""Which of a step's requests have which kernel of the gated scan: every one once, in their order."""
import pytest

from axon_amd.kernels.lib import Kernels


@pytest.mark.parametrize("channels", [1, 64, 512, 2560, 8192])
@pytest.mark.parametrize("lengths", [[], [1], [8], [9], [128], [129], [2000] + [1] * 20, [300, 300, 64, 64, 20, 9, 3, 1], [100] * 100, [5] * 300,
                                     [64] * 4 + [1] * 30, [16] * 16, [17] * 300 + [16] * 3, [129, 128, 17, 16, 9, 8]])
def test_groups_cover_the_requests(lengths, channels):
    groups = Kernels.scan_groups(lengths, channels)
    assert [i for first, end, _ in groups for i in range(first, end)] == list(range(len(lengths)))
    for first, end, longest in groups:
        assert longest in (0, lengths[first])
        assert longest or lengths[first] <= 128            # a thread a channel takes half a microsecond a token
        assert not longest or lengths[end - 1] > 8
        assert not 0 < longest <= 128 or lengths[first] <= 128


def test_lines():
    assert Kernels.scan_groups([2000] + [1] * 20, 2560) == [(0, 1, 2000), (1, 21, 0)]
    assert Kernels.scan_groups([64] * 4 + [1] * 30, 5120) == [(0, 4, 64), (4, 34, 0)]           # the short ones do not count for the longer
    assert Kernels.scan_groups([64] * 31, 2048) == [(0, 31, 64)] and Kernels.scan_groups([64] * 32, 2048) == [(0, 32, 0)]
    assert Kernels.scan_groups([16] * 15, 1024) == [(0, 15, 16)] and Kernels.scan_groups([16] * 16, 1024) == [(0, 16, 0)]
    assert Kernels.scan_groups([200, 100, 12], 64) == [(0, 1, 200), (1, 3, 100)]
