// Host-only C entry points over the launch rules of the device factorisation
// and the tiled solve (host_algos.hpp), built by tests/test_launch_rules.py
// with g++.
#include "host_algos.hpp"

extern "C" int fac_workgroups(int chunks, int levels) {
  return laamd::factor_workgroups(chunks, levels);
}

extern "C" int fac_one_launch(long long rows, long long levels, int lanes,
                              long long eliminations) {
  return laamd::factor_one_launch(rows, levels, lanes, eliminations) ? 1 : 0;
}

extern "C" int tri_touch(long long groups, long long levels, long long record_bytes) {
  return laamd::tile_touch(groups, levels, record_bytes) ? 1 : 0;
}
