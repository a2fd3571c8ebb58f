// Offsets of the row walk (walk_rows) and the shapes that keep them in 32 bits. Plain C++: the
// kernels and a host check use the same expressions.
#pragma once

#include <cstdint>

namespace pdx {
namespace pairk {

constexpr int WALK_U = 4;  // row entries per lane and iteration

// Bytes of the packed positions' buffer resource, which starts one particle early (ids are 1-based).
constexpr uint32_t walk_records(int32_t n) { return ((uint32_t)n + 1u) * 16u; }
// Byte offset of particle id (1-based) in it.
constexpr uint32_t walk_gather(int32_t id) { return (uint32_t)id << 4; }
// Byte offset of a lane's entry in an iteration's rows, and of its u-th entry from there.
constexpr uint32_t walk_lane(int32_t lane, int32_t n, int32_t i) {
  return ((uint32_t)lane * (uint32_t)n + (uint32_t)i) * 4u;
}
constexpr uint32_t walk_step(int32_t u, int32_t lanes, int32_t n) {
  return (uint32_t)u * (uint32_t)lanes * (uint32_t)n * 4u;
}

// Lanes of the walk for `lanes` wanted (split layouts, below zero, have no such offsets): fewer where an
// iteration's rows, WALK_U * lanes * n entries, end beyond 4 GiB; 0, one lane with 64-bit addresses, where
// one lane's do or the packed positions' size is no 32-bit number.
inline int walk_shape(int lanes, int32_t n) {
  constexpr int64_t end = int64_t(1) << 32;
  if (lanes < 0) return lanes;
  while (lanes > 1 && 4ll * WALK_U * lanes * n >= end) lanes >>= 1;
  return lanes == 1 && (4ll * WALK_U * n >= end || 16ll * ((int64_t)n + 1) >= end) ? 0 : lanes;
}

}  // namespace pairk
}  // namespace pdx
