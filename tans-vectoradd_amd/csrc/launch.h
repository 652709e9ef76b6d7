// Launch rules that depend on the device's CU count, in plain C++.
#ifndef TANS_LAUNCH_H
#define TANS_LAUNCH_H

#include <stdint.h>

// Compute units of the current device (0 if they cannot be queried).
extern "C" int tans_internal_cu_count();   // kernels.hip

namespace tans_launch {

// Waves of each workgroup that decode, for `units` wave-sized pieces of work
// (a wave takes one at a time) on `cus` workgroups, one per CU: as few as
// keep the number of rounds.  The 16 waves of a full workgroup share the
// CU's issue slots, and a wave with a SIMD to itself decodes a tile in 0.85
// us instead of 1.9, so pieces that do not fill the chip are spread over all
// CUs rather than packed into a few.  Fused add, 1024 per lane, 16 waves per
// workgroup against this rule: 256 groups 91.6 -> 61.6 us, 1024 groups 93.8
// -> 67 us, 2048 groups 96.4 -> 78 us (with the kernels for few waves, see
// fused_add_kernel, 50, 54 and 70 us), 5000 groups (two rounds of 10 waves per
// CU, not 16 and then 16 on a fifth of the CUs) 210 -> 180 us.
//
// Half of kDecWaves or fewer means one round: ceil(units / waves) workgroups are
// then no more than the CUs, and a wave takes one piece or none.  (From two
// rounds on, more than (rounds - 1) / rounds of kDecWaves are needed.)  The
// kernels for few waves rely on it.
constexpr int kDecWaves = 16;   // waves of a full decoding workgroup, one per CU
inline int spread_waves(int64_t units, int cus) {
    const int64_t per_round = (int64_t)cus * kDecWaves;
    const int64_t rounds = (units + per_round - 1) / per_round;
    return (int)((units + cus * rounds - 1) / (cus * rounds));
}

// Whether the GPU encoder's walk of G groups of N elements per lane loads whole
// lines (enc_walk_kernel's LINES): rows of whole 128-byte lines, and rounds of
// 16 groups per CU that are at least three quarters full in all (the other
// kernel's smaller workgroups fill a part round better).  Calls with it against
// without on 256 CUs, 1024 per lane: 256 groups 121 / 90 us, 2048 groups 134 /
// 128, 4096 groups 185 / 205, 4160 groups 249 / 226, 6250 groups 291 / 315, 8192
// groups 360 / 398; 62500 groups of 128 per lane 404 / 422 us.
constexpr int64_t kLineBytes = 128;
constexpr int64_t kLineWaves = 16;   // groups (waves) of a workgroup, one per CU
inline bool whole_lines(int64_t G, int64_t N, int cus) {
    const int64_t round = kLineWaves * cus;
    const int64_t rounds = (G + round - 1) / round;
    return N % kLineBytes == 0 && 4 * G >= 3 * rounds * round;
}

}  // namespace tans_launch

#endif  // TANS_LAUNCH_H
