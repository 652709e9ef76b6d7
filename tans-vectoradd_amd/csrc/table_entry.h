// Entries of the decode table, in plain C++ so that the bound every decoder
// rests on (an entry as it lies in LDS never leads outside the table) is checked
// on the CPU for every input.
#ifndef TANS_TABLE_ENTRY_H
#define TANS_TABLE_ENTRY_H

#include "schedule.h"

namespace tans_table {

// word0: nb in bits 7:0 and 31:27, the symbol's exponents in bits 14:11 and
// 22:19; word1: (base - L) * 8, the byte offset of the next state's entry for
// stream bits 0.
struct Entry {
    uint32_t x, y;
};

TANS_SCHED_FN int floor_log2(uint32_t v) { return 31 - __builtin_clz(v); }

// The entry of a slot of `sym` (below 256, or 16 with a 2^11-state table) that is
// its rank-th in slot order, f being the symbol's frequency; as the host
// builder (codec.cpp) writes it where rank < f.  Any f and rank are taken.
TANS_SCHED_FN Entry entry(int log2L, uint32_t sym, uint32_t f, uint32_t rank) {
    const uint32_t L = 1u << log2L;
    const uint32_t xp = f + rank;
    const int top = xp ? floor_log2(xp) : log2L;
    const int nb = top < log2L ? log2L - top : 0;
    const uint32_t ex =
        log2L == tans_sched::kTripleLog2L ? sym << 11 : ((sym >> 4) << 11) | ((sym & 0xFu) << 19);
    return Entry{(uint32_t)nb | ex | ((uint32_t)nb << 27), ((xp << nb) - L) * 8u};
}

// A table entry as the decoders keep it in LDS: one that would step outside
// the table (nb > log2L or base + 2^nb > 2L), or read more bits than the refill
// schedule allows (nb > 10 in a 2^11-state table), becomes a harmless one.
// packed: the packed-layout decoders' word0, which keeps nb in bits 4:0 and
// moves the two exponents 8 bits up (bits 22:19 and 30:27), so that bits 15:0
// of a sum of word0s are the sum of their nb.
TANS_SCHED_FN Entry lds_entry(int log2L, bool packed, Entry e) {
    const uint32_t max_nb =
        log2L == tans_sched::kTripleLog2L ? tans_sched::kTripleMaxNb : (uint32_t)log2L;
    const uint32_t nb = e.x & 0xFFu;
    const uint32_t base = e.y >> 3;
    if (nb > max_nb || (e.x >> 27) != nb || (e.y & 7u) || base + (1u << nb) > (1u << log2L))
        e = Entry{e.x & 0x07FFFF00u, 0u};
    if (packed) e.x = (e.x & 0x1Fu) | ((e.x & 0x007FF800u) << 8);
    return e;
}

}  // namespace tans_table

#endif  // TANS_TABLE_ENTRY_H
