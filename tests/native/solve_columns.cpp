// Columns of one solve whose lane offsets fit 32 bits (csrc/plan.hpp).  Prints "ok".
#include <cstdio>

#include "plan.hpp"

int main() {
  const int64_t two32 = (int64_t)1 << 32;
  for (int64_t n : {1ll, 200000ll, 960000ll, 8521760ll, 8521761ll, 8600000ll, 9000000ll, 17000000ll, 100000000ll,
                    500000000ll}) {
    const int c = spde::solve_columns(n);
    // the furthest lane of a tile of c columns (at most 64): its last column, 12 rows on
    const int64_t last = 8 * n * ((c < 64 ? c : 64) - 1) + 96;
    const bool fits = last < two32, most = c >= 64 || 8 * n * c + 96 >= two32;
    if (c < 1 || !fits || !most || (c >= 64 && c != INT32_MAX)) {
      std::printf("n %lld: %d columns\n", (long long)n, c);
      return 1;
    }
  }
  std::printf("ok\n");
}
