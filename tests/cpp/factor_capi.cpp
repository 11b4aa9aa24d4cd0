// Host-only C entry points over the launch rules of the device factorisation
// (host_algos.hpp), built by tests/test_factor_rules.py with g++.
#include "host_algos.hpp"

extern "C" int fac_workgroups(int chunks, int levels) {
  return laamd::factor_workgroups(chunks, levels);
}

extern "C" int fac_one_launch(long long rows, long long levels, int lanes,
                              long long eliminations) {
  return laamd::factor_one_launch(rows, levels, lanes, eliminations) ? 1 : 0;
}
