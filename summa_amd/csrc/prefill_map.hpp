// Which workgroup of the prefill attention takes which (KV head of a sequence,
// query head, row tile). Host and device, so that the map can be walked on the CPU.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace sm {

// Workgroups go to the 8 XCDs in turn. A group is the `per` workgroups that share a
// KV head's K and V. Whole eights of groups take one XCD each, whose L2 then reads
// that K and V from memory once. The rest, fewer than eight groups, are dealt out
// over all XCDs, each group to as few of them as keeps the XCDs even: 4 groups to 2
// XCDs each, 6 in threes to 4, an odd number all to 8. One sequence, 16 heads of 128,
// causal, us with every group on one XCD / so / in the order of rows, heads and
// sequences (a kernel with 16-query waves): 4 KV heads, 4096 positions 228 / 151 / 230;
// 2, 8192 1540 / 440 / 842; 1, 4096 719 / 144 / 225; 9 sequences of 512, 1 KV head 45 / 39
// / 56.
// (32 bits hold every count: the queries and keys of 2^31 workgroups fit no card.)
struct PrefillMap {
  uint32_t groups, per;
  uint32_t whole;       // groups on an XCD of their own
  uint32_t sets, span;  // the rest: `sets` sets of `span` XCDs (sets * span = 8)

  __host__ __device__ PrefillMap(uint32_t groups_, uint32_t per_) : groups(groups_), per(per_) {
    const uint32_t rest = groups % 8;
    whole = groups - rest;
    sets = rest == 0 ? 8 : rest == 4 ? 4 : rest % 2 == 0 ? 2 : 1;
    span = 8 / sets;
  }
  __host__ __device__ int64_t workgroups() const {
    const int64_t rest = (int64_t)((groups - whole) / sets) * per;  // a set's
    return 8 * ((int64_t)(whole / 8) * per + (rest + span - 1) / span);
  }
  // Workgroup `wg` < workgroups(): its group and its place 0 .. per - 1 in it; false
  // where there is nothing to do.
  __host__ __device__ bool at(uint32_t wg, uint32_t& group, uint32_t& place) const {
    const uint32_t xcd = wg % 8, i = wg / 8;
    if (i < whole / 8 * per) {
      group = i / per * 8 + xcd;
      place = i % per;
      return true;
    }
    const uint32_t n = (groups - whole) / sets;  // groups of a set
    const uint32_t u = (i - whole / 8 * per) * span + xcd % span;
    if (u >= n * per) return false;
    group = whole + xcd / span * n + u / per;
    place = u % per;
    return true;
  }
};

}  // namespace sm
