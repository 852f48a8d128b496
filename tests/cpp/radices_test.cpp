// CPU test of the mixed-radix passes' stage radices (fishfry_amd/csrc/ff_mixplan.cpp):
// for every length the product is the length, radices above 13 are prime and come
// last, and lengths without a prime factor above 13 have none of them.  The
// device tables are link stand-ins that are never called.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "ff_internal.hpp"
#include "ff_mixed.hpp"

namespace ff {
const void* table_twiddle(int, int) { return nullptr; }
const void* table_built(int, int, int, const TableBuilder&) { return nullptr; }
void twiddle_ld(long long, long long, long double&, long double&) {}
}  // namespace ff

#define REQUIRE(c)                                                                  \
  do {                                                                              \
    if (!(c)) {                                                                     \
      std::fprintf(stderr, "FAILED %s for n = %d (line %d)\n", #c, n, __LINE__);    \
      std::exit(1);                                                                 \
    }                                                                               \
  } while (0)

static bool prime(int v) {
  for (int p = 2; p * p <= v; ++p)
    if (v % p == 0) return false;
  return v > 1;
}

int main() {
  for (int n = 2; n <= 16384; ++n) {
    int largest = 1;
    for (int v = n, p = 2; v > 1; ++p)
      while (v % p == 0) largest = p, v /= p;
    const std::vector<int> rs = ff::mix_radices(n);
    if (largest > ff::kMixMaxDense) {
      REQUIRE(rs.empty());
      continue;
    }
    if (rs.empty()) {  // too many stages
      long long least = 1;
      for (int k = 0; k < ff::kMixStages; ++k) least *= 2;
      REQUIRE(n > least);
      continue;
    }
    long long product = 1;
    bool dense = false;
    for (int r : rs) {
      product *= r;
      if (r > 13) {
        REQUIRE(prime(r));
        dense = true;
      } else {
        REQUIRE(!dense);
      }
    }
    REQUIRE(product == n);
    REQUIRE(dense == (largest > 13));
    // ascending dense radices, descending small ones
    REQUIRE(std::is_sorted(rs.begin(), std::find_if(rs.begin(), rs.end(), [](int r) { return r > 13; }),
                           [](int a, int b) { return a > b; }));
    REQUIRE(std::is_sorted(std::find_if(rs.begin(), rs.end(), [](int r) { return r > 13; }), rs.end()));
  }
  std::printf("radices ok\n");
  return 0;
}
