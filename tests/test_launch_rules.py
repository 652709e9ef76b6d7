"""Launch rules that depend on how many CUs the device has: the lines they
draw follow the CU count, not one card's 256.  The C++ rules (csrc/launch.h)
are plain C++ and run here from a small library built with g++."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "tans-vectoradd_amd", "csrc")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("launch")
    src = d / "rules.cpp"
    src.write_text('''#include "launch.h"
extern "C" int whole_lines(int64_t G, int64_t N, int cus) {
    return tans_launch::whole_lines(G, N, cus);
}
extern "C" int spread_waves(int64_t units, int cus) { return tans_launch::spread_waves(units, cus); }
''')
    out = d / "librules.so"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                    str(src), "-o", str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    lib.whole_lines.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    lib.spread_waves.argtypes = [ctypes.c_int64, ctypes.c_int]
    return lib


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


@pytest.mark.parametrize("cus", [32, 128, 256, 304])
def test_encoder_loads_lines_in_rounds_of_this_device(rules, cus):
    """Whole-line loads from three quarters of the device's rounds (16 groups
    per CU) on, for rows of whole 128-byte lines only."""
    round_ = 16 * cus
    for rounds in (1, 2, 7):
        full, least = rounds * round_, -(-3 * rounds * round_ // 4)
        first = max(least, (rounds - 1) * round_ + 1)   # the fewest groups of this many rounds
        assert rules.whole_lines(full, 128, cus) and rules.whole_lines(first, 4096, cus)
        if first == least:
            assert not rules.whole_lines(least - 1, 128, cus)
        assert not rules.whole_lines(full, 192, cus) and not rules.whole_lines(full, 130, cus)
    assert not rules.whole_lines(1, 1024, cus)
    assert not rules.whole_lines(round_ + 1, 1024, cus)   # half of two rounds


@pytest.mark.parametrize("cus", [1, 32, 256, 304])
def test_waves_are_as_few_as_keep_the_rounds(rules, cus):
    """1..16 waves, the rounds of 16-wave workgroups, no wave fewer; and up to 8
    waves one round with no more workgroups than CUs, so that the kernels for
    few waves, which take one piece per wave, leave none over."""
    full = 16 * cus
    around = (1, 2, cus, 8 * cus, full, 2 * full, 3 * full, 17 * full)
    for units in sorted({u + d for u in around for d in (-1, 0, 1, 5)} - {0, -1}):
        w = rules.spread_waves(units, cus)
        rounds = -(-units // full)
        assert 1 <= w <= 16
        assert -(-units // (w * cus)) == rounds
        assert w == 1 or -(-units // ((w - 1) * cus)) > rounds
        if w <= 8:
            assert rounds == 1 and -(-units // w) <= cus
