// The source offsets of the general limb split on the host (built by
// tests/test_split_offsets.py with g++ -fsanitize=undefined): against a
// counter over the modes, at and past the end, and for modes of extent zero.
#include <cstdio>
#include <vector>

#include "tamx_offsets.hpp"

static int check(const std::vector<int32_t>& ext, const std::vector<int64_t>& str) {
  const int n = (int)ext.size();
  int count = 1, bad = 0;
  for (int e : ext) count *= e;
  std::vector<int> idx(n, 0);
  for (int x = 0; x < count + 128; ++x) {
    int64_t want = 0;
    for (int d = 0; d < n && x < count; ++d) want += idx[d] * str[d];
    if (tamx::split::mixed_radix_offset(x, count, n, ext.data(), str.data()) != want) ++bad;
    for (int d = n - 1; d >= 0 && ++idx[d] == ext[d]; --d) idx[d] = 0;
  }
  return bad;
}

int main() {
  int bad = 0;
  bad += check({7}, {3});
  bad += check({3, 5}, {1, 3});
  bad += check({2, 3, 4, 5}, {1, 200, 10, 0});
  bad += check({0}, {1});
  bad += check({3, 0}, {1, 3});
  bad += check({0, 3}, {1, 3});
  bad += check({2, 0, 0, 4}, {1, 2, 3, 4});
  std::printf(bad ? "%d offsets differ\n" : "OFFSETS OK\n", bad);
  return bad != 0;
}
