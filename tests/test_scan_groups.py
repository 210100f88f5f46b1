"""Which of a step's requests have which kernel of the gated scan: every one once, in their order."""
import pytest

from axon_amd.kernels.lib import Kernels


@pytest.mark.parametrize("channels", [1, 64, 512, 2560, 8192])
@pytest.mark.parametrize("lengths", [[], [1], [8], [9], [128], [129], [2000] + [1] * 20, [300, 300, 64, 64, 20, 9, 3, 1], [100] * 100, [5] * 300,
                                     [64] * 4 + [1] * 30, [16] * 16, [17] * 300 + [16] * 3, [129, 128, 17, 16, 9, 8]])
def test_groups_cover_the_requests(lengths, channels):
    groups = Kernels.scan_groups(tuple(lengths), channels)
    assert [i for first, end, _ in groups for i in range(first, end)] == list(range(len(lengths)))
    for first, end, fed in groups:
        assert fed or lengths[first] <= 128            # a thread a channel takes half a microsecond a token
    assert [fed for _, _, fed in groups] in ([], [True], [False], [True, False])


def test_lines():
    groups = lambda lengths, channels: Kernels.scan_groups(tuple(lengths), channels)
    assert groups([2000] + [1] * 20, 2560) == ((0, 21, True),) and groups([512] + [1] * 100, 2560) == ((0, 1, True), (1, 101, False))
    assert groups([300, 100, 50, 20, 8, 4, 1], 2560) == ((0, 7, True),) and groups([300, 20], 5120) == ((0, 2, True),)
    assert groups([64] * 16 + [1] * 16, 5120) == ((0, 16, True), (16, 32, False)) and groups([64] * 16 + [1] * 16, 512) == ((0, 32, True),)
    assert groups([32] * 64, 2560) == ((0, 64, False),) and groups([32] * 64, 512) == ((0, 64, True),)
    assert groups([5] * 300, 512) == ((0, 300, False),) and groups([12, 9, 5], 2560) == ((0, 3, True),)
