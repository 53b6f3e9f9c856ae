// When the router preprocess runs in one workgroup: shared by the launcher and the host side, which then allocates no scratch.
#pragma once
#include <stdint.h>

constexpr int kRouteSmallRounds = 8;             // rounds of 1024 ids
constexpr int64_t kRouteSmallLds = 60 << 10;     // bytes of counts, [ids / 64][E], and totals
inline int64_t aamd_route_small_lds(int64_t n, int64_t E) { return ((n + 63) / 64 + 1) * E * (int64_t)sizeof(int); }
inline bool aamd_route_one_workgroup(int64_t n, int64_t E) {
  return n <= kRouteSmallRounds * 1024 && aamd_route_small_lds(n, E) <= kRouteSmallLds;
}
// Whether it should, where there is scratch for the other forms: one workgroup takes 2.2 us and 1 to 1.7 for every 1024 ids, two
// launches of a workgroup per 1024 ids 6 to 8 in all, and 10 with hundreds of experts, whose counts each of them adds up.  The line lies where
// both take the same.  One and two, us: 1 expert, 3300 ids 5.1 and 6.2, 4600 6.1 and 6.2, 5000 6.7 and 6.2; 2, 3300 5.4 and 6.1, 3900 6.0 and
// 6.1, 4300 6.4 and 6.1; 3, 3700 6.1 and 6.2; 4, 3500 5.9 and 6.1; replayed in a graph: 8, 3328 6.2 and 6.2, 4096 7.0 and 6.2, 8192 12.1 and
// 6.7; 60, 3328 6.9 and 7.0, 4096 8.0 and 6.8, 8192 14.2 and 7.4; 128, 3584 7.9 and 7.8, 4096 8.8 and 7.7; 192, 3584 8.4 and 8.6, 4096 9.4 and
// 8.6; 236, 3584 8.6 and 9.4, 4096 9.8 and 9.2; 300, 3073 8.7 and 10.4.
inline bool aamd_route_takes_scratch(int64_t n, int64_t E) { return n > 3200 + 3 * E + 1400 / (E < 1 ? 1 : E) || !aamd_route_one_workgroup(n, E); }
