// ensure_arrays (tgh_scratch.hpp) on the CPU with an allocator that fails once:
// the failed call reports it and leaves the missing array null, the next call
// makes what is missing and keeps what is there.
#include "../../treegeneralizedharmonic.jl_amd/csrc/tgh_scratch.hpp"

#include <cstdio>

int main() {
  static double mem[3];
  for (int fail_at = 0; fail_at < 3; ++fail_at) {
    double* p[3] = {nullptr, nullptr, nullptr};
    int calls = 0, next = 0;
    auto get = [&](double** at, size_t bytes) {
      if (bytes != 8) return 2;
      *at = &mem[next];
      if (calls++ == fail_at) return 1;  // an array that could be made but not cleared
      ++next;
      return 0;
    };
    auto ensure = [&] { return tgh::ensure_arrays({{&p[0], 8}, {&p[1], 8}, {&p[2], 8}}, get); };
    if (ensure() != 1) return 10;
    for (int i = 0; i < 3; ++i)
      if ((p[i] != nullptr) != (i < fail_at)) return 11;
    double* kept = p[0];
    if (ensure() != 0 || !p[0] || !p[1] || !p[2]) return 12;
    if (fail_at > 0 && p[0] != kept) return 13;
    if (calls != 4 || ensure() != 0 || calls != 4) return 14;  // nothing is made twice
  }
  std::printf("ok\n");
  return 0;
}
