// Growth of a backend's device scratch, apart from the calls that allocate it.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace spiral {

struct Scratch {
  uint8_t* base = nullptr;
  size_t size = 0;
};

// Makes s hold `need` bytes; where alloc(n) (null on failure) has no room for
// them, `least` bytes or as many as s had. False: not even those, and s is empty.
// The old memory goes first: a scratch of hundreds of MiB is not held twice.
template <typename Alloc, typename Release>
bool grow(Scratch& s, size_t need, size_t least, Alloc alloc, Release release) {
  if (need <= s.size) return true;
  if (least < s.size) least = s.size;
  if (s.base != nullptr) release(s.base);
  s = Scratch{};
  const size_t sizes[2] = {need, least};
  for (int i = 0; i < (least < need ? 2 : 1); ++i) {
    void* p = alloc(sizes[i]);
    if (p == nullptr) continue;
    s.base = static_cast<uint8_t*>(p);
    s.size = sizes[i];
    return true;
  }
  return false;
}

}  // namespace spiral
