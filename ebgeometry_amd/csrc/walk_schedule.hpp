// How far the stack of a long walk is spread before it is handed on (HandOn).
#pragma once

#include <algorithm>
#include <cstdint>

namespace ebgpu {

constexpr uint32_t kHandBudget[2] = {150, 60}; // HandOn::budget (measured: api.cpp)
constexpr int      kHandSpread[2] = {48, 32};  // HandOn::spread, at most

// HandOn::spread[stage] for stacks of `capacity` entries. A wavefront that finds no room after it has
// spread its stack goes on from it, depth-first, and must not need more than the capacity then. Spreading
// ends at no more than spread + 2 entries, and the ones above the lowest 4, which a walk from the root
// has room for too, lie at least two levels below the root; deep_need (WalkTree) is what the walk from one
// of those needs. 48 entries on trees of 327,680 faces with leaves of 1 and 2 reached 65 to 67 of 64.
inline int hand_spread(int stage, int capacity, int deep_need)
{
  return std::max(0, std::min(kHandSpread[stage], capacity - 1 - deep_need));
}

// Whether a walk of a tree of `visits` nodes and leaves can use up its budget. If not, its calls need none of
// the launches that take up what was handed on (100 queries on 80 faces: 61 us with them, 46 without; 1
// query 63 and 37).
inline bool can_hand_on(uint64_t visits, uint32_t budget) { return visits > budget; }

// Whether HandOn's 32-bit counter of slots can count `walks` requests (all of them, granted or not).
inline bool hand_counts_fit(uint64_t walks) { return walks <= 0xFFFFFFFFull; }

} // namespace ebgpu
