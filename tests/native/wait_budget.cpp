// The budget of the factorisation's bounded waits (csrc/wait.hpp).  Prints "ok".
#include <cstdio>

#include "wait.hpp"

int main() {
  using spde::kSpinLimit;
  spde::WaitBudget w;
  // many healthy waits of one block, together far beyond the limit of one
  const int polls = 1000, waits = 3 * (kSpinLimit / polls);
  for (int i = 0; i < waits; ++i) {
    w.begin();
    for (int k = 0; k < polls; ++k)
      if (w.spent()) {
        std::printf("healthy waits added up to a stall at wait %d\n", i);
        return 1;
      }
  }
  // a wait in vain ends right after the limit, also after others
  w.begin();
  int n = 0;
  while (!w.spent()) ++n;
  if (n != kSpinLimit) {
    std::printf("a wait in vain ended after %d polls\n", n);
    return 1;
  }
  std::printf("ok\n");
}
