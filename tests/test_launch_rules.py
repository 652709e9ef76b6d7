"""Launch rules that depend on how many CUs the device has: the lines they
draw follow the CU count, not one card's 256."""
import pytest


@pytest.mark.parametrize("cus", [32, 128, 256, 304])
def test_decode_tables_are_built_by_rounds_of_this_device(cus):
    """A decode's workgroups build their own tables for two rounds of 32 groups
    per CU and read one built before from the next group on; columns of one or
    two tiles run in one round at any lane count."""
    from rans_vectoradd import _C
    lanes = 2 * 32 * 64 * cus
    for N in (34, 48, 1024):
        assert _C._builds_each(lanes, N, cus)
        assert not _C._builds_each(lanes + 1, N, cus)
    for N in (2, 16, 32):
        assert _C._builds_each(100 * lanes, N, cus)
