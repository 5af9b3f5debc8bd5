// Bounded waits of the kernels whose blocks hand tiles to each other.
#pragma once

namespace spde {

// Polls before a wait gives up (seconds; a healthy wait takes microseconds).
constexpr int kSpinLimit = 1 << 22;

// The polls of one wait, and whether an earlier wait gave up.  Each wait has the
// whole limit: a block waits thousands of times in a launch, and healthy waits
// must not add up to a stall.
struct WaitBudget {
  int spins = 0;
  bool gave_up = false;
  constexpr void begin() { spins = 0; }
  // counts a poll in vain; true when the limit is passed
  constexpr bool spent() { return ++spins > kSpinLimit; }
};

}  // namespace spde
