// Device arrays that are allocated at first use, several at a time.
#pragma once
#include <cstddef>
#include <initializer_list>

namespace tgh {

struct ScratchArray {
  double** at;
  size_t bytes;
};
// Makes every array of the list that is not there yet: get(at, bytes) sets *at
// and returns 0, or returns an error code, which ends the list. Each array is
// looked at by itself, so that a call after one that found no memory half way
// goes on where that one stopped and never takes a missing array for made.
template <class Get>
int ensure_arrays(std::initializer_list<ScratchArray> arrays, const Get& get) {
  for (const ScratchArray& a : arrays) {
    if (*a.at) continue;
    const int rc = get(a.at, a.bytes);
    if (rc) {
      *a.at = nullptr;
      return rc;
    }
  }
  return 0;
}

}  // namespace tgh
