"""Which element patterns go by ranges (host logic of libspion_hip.so, spion_debug_remainder_by_ranges: no device needed)."""
import pytest

from spion_amd import _lib


def _by_ranges(heads, length, per_row, cus=256):
    return _lib.core().spion_debug_remainder_by_ranges(heads, length, int(per_row * length), cus)


# heads, length, entries a row, whether ranges were measured as the faster way by more than a fifth (forward and backward)
@pytest.mark.parametrize("heads,length,per_row,ranges", [
    (128, 512, 2, 1), (100, 512, 48, 1), (64, 1024, 16, 1), (64, 1024, 128, 1), (64, 1536, 300, 1), (32, 2048, 4, 1), (64, 2048, 128, 1),
    (40, 2048, 16, 1), (12, 3072, 300, 1), (16, 4096, 128, 1), (64, 4096, 2, 1), (64, 4096, 128, 1), (8, 8192, 128, 1), (32, 8192, 128, 1),
    (16, 16384, 128, 1), (4, 16384, 300, 1), (4, 32768, 300, 1),
    (16, 512, 16, 0), (32, 512, 32, 0), (16, 1024, 32, 0), (8, 1024, 300, 0), (8, 2048, 16, 0), (4, 4096, 2, 0), (4, 4096, 128, 0),
    (8, 4096, 48, 0), (2, 8192, 64, 0), (8, 8192, 16, 0), (12, 8192, 4, 0), (1, 16384, 16, 0), (1, 16384, 128, 0), (4, 16384, 32, 0),
    (16, 16384, 4, 0), (1, 32768, 128, 0), (4, 32768, 32, 0)])
def test_the_faster_way_is_taken(heads, length, per_row, ranges):
    assert _by_ranges(heads, length, per_row) == ranges


def test_the_index_is_bounded_by_the_pattern():
    """A list by ranges has L / 512 offsets for every row and every column: a few tens and a fraction of the entries."""
    for heads in (1, 2, 5, 16, 64, 300, 4096):
        for log in range(9, 19):
            for length in (1 << log, (1 << log) + (32 if log < 18 else -32)):
                for per_row in (1, 4, 16, 64, 256, 1024, 4096):
                    if per_row <= length and _by_ranges(heads, length, per_row):
                        assert -(-length // 512) <= 16 + 0.25 * per_row, (heads, length, per_row)


def test_limits():
    core = _lib.core()
    assert _by_ranges(64, 480, 16) == 0 and _by_ranges(64, (1 << 18) + 32, 4096) == 0
    assert core.spion_debug_remainder_by_ranges(64, 4096, 0, 256) == 0  # an empty remainder
    # {dS, P} of an entry are found by a signed 32-bit byte offset, 8 bytes an entry
    assert [core.spion_debug_remainder_by_ranges(16, 32768, n, 256) for n in ((1 << 28) - 1, 1 << 28, (1 << 29) - 1)] == [1, 0, 0]
    for bad in ((0, 4096, 1, 256), (64, 0, 1, 256), (64, 4096, 1, 0)):
        assert core.spion_debug_remainder_by_ranges(*bad) == -1
