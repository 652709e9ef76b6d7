// Launch rules that depend on the device's CU count, in plain C++.
#ifndef TANS_LAUNCH_H
#define TANS_LAUNCH_H

#include <stdint.h>

// Compute units of the current device (0 if they cannot be queried).
extern "C" int tans_internal_cu_count();   // kernels.hip

namespace tans_launch {

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
