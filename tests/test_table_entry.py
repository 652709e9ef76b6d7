"""The decode table's entries (csrc/table_entry.h, built here with g++): as the
decoders keep them in LDS they lead nowhere outside the table and read no more
bits than the refill schedule allows, whatever spread and frequencies they come
from, and those of a consistent pair are the host builder's."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "tans-vectoradd_amd", "csrc")

SOURCE = """#include "table_entry.h"
using namespace tans_table;

static bool in_range(int log2L, Entry e, bool packed) {
    const uint32_t nb = packed ? e.x & 0x1Fu : e.x & 0xFFu;
    const uint32_t max_nb = log2L == tans_sched::kTripleLog2L ? tans_sched::kTripleMaxNb : log2L;
    // the last entry a step can reach: offset + 8 * (2^nb - 1)
    return nb <= max_nb && e.y % 8 == 0 && (uint64_t)e.y / 8 + (1u << nb) <= (1u << log2L) &&
           (packed || e.x >> 27 == nb);
}

// entries out of range among those of frequency f and every rank a slot can have
extern "C" int64_t bad_entries(int log2L, uint32_t f) {
    int64_t bad = 0;
    const uint32_t syms = log2L == tans_sched::kTripleLog2L ? 16 : 256;
    for (uint32_t rank = 0; rank < (1u << log2L); rank++) {
        const Entry e = entry(log2L, rank % syms, f, rank);
        bad += !in_range(log2L, lds_entry(log2L, false, e), false);
        bad += !in_range(log2L, lds_entry(log2L, true, e), true);
    }
    return bad;
}

// ... and of any two words
extern "C" int64_t bad_words(int log2L, uint32_t x, uint32_t y) {
    const Entry e{x, y};
    return !in_range(log2L, lds_entry(log2L, false, e), false) +
           !in_range(log2L, lds_entry(log2L, true, e), true);
}

// the table of a spread, ranks by counting
extern "C" void build(int log2L, const int32_t* spread, const int32_t* freqs, uint32_t* table) {
    uint32_t seen[256] = {};
    for (int i = 0; i < 1 << log2L; i++) {
        const uint32_t s = (uint32_t)spread[i];
        const Entry e = entry(log2L, s, (uint32_t)freqs[s], seen[s]++);
        const Entry kept = lds_entry(log2L, false, e);
        table[2 * i] = kept.x;
        table[2 * i + 1] = kept.y;
    }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("entry")
    (d / "entry.cpp").write_text(SOURCE)
    out = d / "libentry.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-shared", "-fPIC", f"-I{CSRC}",
                    str(d / "entry.cpp"), "-o", str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    lib.bad_entries.argtypes = [ctypes.c_int, ctypes.c_uint32]
    lib.bad_words.argtypes = [ctypes.c_int, ctypes.c_uint32, ctypes.c_uint32]
    lib.bad_entries.restype = lib.bad_words.restype = ctypes.c_int64
    return lib


@pytest.mark.parametrize("log2L", [12, 11])
def test_entries_of_any_frequency_stay_in_the_table(lib, log2L):
    """Every rank a slot can have (0 .. L - 1) at frequencies around 0, the
    powers of two, the table size and the ends of 32 bits (negative ones among
    them): a spread holds no other pairs of the two."""
    L = 1 << log2L
    freqs = set(range(L + 2))
    freqs |= {(1 << b) + d for b in range(32) for d in (-1, 0, 1)}
    freqs |= {-d % (1 << 32) for d in (1, 2, L - 1, L, L + 1)}
    assert sum(lib.bad_entries(log2L, f) for f in freqs) == 0


@pytest.mark.parametrize("log2L", [12, 11])
def test_any_words_stay_in_the_table(lib, log2L):
    g = np.random.default_rng(log2L)
    for x, y in g.integers(0, 1 << 32, (20000, 2), dtype=np.uint64).tolist():
        nb = x % 14    # plausible entries too: nb in both places, a small offset
        for w0, w1 in ((x, y), (nb | nb << 27, y), (nb | nb << 27, y % (10 << log2L) // 8 * 8)):
            assert lib.bad_words(log2L, w0 & 0xFFFFFFFF, w1) == 0, (w0, w1)


@pytest.mark.parametrize("alphabet,log2L", [("pair", 12), ("nibble", 11)])
@pytest.mark.parametrize("steep", [0.0, 0.5, 2.0])
def test_entries_of_a_consistent_pair_are_the_host_builders(lib, alphabet, log2L, steep):
    from rans_vectoradd import tans_codec as T
    f = T.symbol_freqs(2.0 ** (-steep * np.arange(16)), alphabet).astype(np.int32)
    sp = T.build_spread(f).astype(np.int32)
    got = np.empty(2 << log2L, dtype=np.uint32)
    lib.build(log2L, sp.ctypes.data_as(ctypes.c_void_p), f.ctypes.data_as(ctypes.c_void_p),
              got.ctypes.data_as(ctypes.c_void_p))
    want = T.build_decode_table(sp, f).numpy().view(np.uint32).reshape(-1)
    assert np.array_equal(got, want)
