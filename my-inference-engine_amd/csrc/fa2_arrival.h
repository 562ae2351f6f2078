// Arrival counts of a launch whose last work-group finishes what the others left.
#pragma once

#include <cstdint>

namespace mi_fa2 {

// What work-group i of n adds to the counter: the weights of a launch add up to 0 (mod 2^32) and no
// proper part of them does, so the one whose add makes the counter 0 is the last, and the counter is
// ready for the next launch as it stands.  Launches that overlap on one counter, against the contract,
// may each miss their last work-group, but leave it at 0 all the same: the damage ends with them.
constexpr uint32_t arrival_weight(uint32_t i, uint32_t n) { return i == 0 ? 1u - n : 1u; }

}  // namespace mi_fa2
