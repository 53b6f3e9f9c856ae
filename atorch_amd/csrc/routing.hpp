// When the router preprocess runs in one workgroup: shared by the launcher and the host side, which then allocates no scratch.
#pragma once
#include <stdint.h>

constexpr int kRouteSmallRounds = 8;             // rounds of 1024 ids
constexpr int64_t kRouteSmallLds = 60 << 10;     // bytes of counts, [ids / 64][E], and totals
inline int64_t aamd_route_small_lds(int64_t n, int64_t E) { return ((n + 63) / 64 + 1) * E * (int64_t)sizeof(int); }
inline bool aamd_route_one_workgroup(int64_t n, int64_t E) {
  return n <= kRouteSmallRounds * 1024 && aamd_route_small_lds(n, E) <= kRouteSmallLds;
}
