// When the router preprocess runs in one workgroup: shared by the launcher and the host side, which then allocates no scratch.
#pragma once
#include <stdint.h>

constexpr int kRouteSmallRounds = 8;             // rounds of 1024 ids
constexpr int64_t kRouteSmallLds = 60 << 10;     // bytes of counts, [ids / 64][E], and totals
inline int64_t aamd_route_small_lds(int64_t n, int64_t E) { return ((n + 63) / 64 + 1) * E * (int64_t)sizeof(int); }
inline bool aamd_route_one_workgroup(int64_t n, int64_t E) {
  return n <= kRouteSmallRounds * 1024 && aamd_route_small_lds(n, E) <= kRouteSmallLds;
}
// Whether it should, where there is scratch for the other forms: one workgroup takes 2.2 us and 1.25 to 1.7 for every 1024 ids, two
// launches of a workgroup per 1024 ids 6.5 to 8 in all.  One and two, us, replayed in a graph: 8 experts, 3072 ids 6.1 and 6.5, 4096
// 7.3 and 6.5, 8192 12.4 and 7.0; 60 experts 6.8 and 7.3, 8.3 and 7.2, 14.6 and 7.7; 128 experts 7.4 and 8.1, 9.2 and 8.2.
constexpr int64_t kRouteSmallIds = 3072;
inline bool aamd_route_takes_scratch(int64_t n, int64_t E) { return n > kRouteSmallIds || !aamd_route_one_workgroup(n, E); }
