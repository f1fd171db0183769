// overlap.hpp -- whether buffers of a call share memory (host side). The kernels that join several of
// the reference's dispatches in one launch read and write in no order between workgroups, so they run
// only where what they write is apart from what they read; other calls go one dispatch after another.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <initializer_list>

namespace mla {

struct Span {
  const void* p;
  size_t bytes;
};

inline bool overlap(const Span& a, const Span& b) {
  const uintptr_t x = (uintptr_t)a.p, y = (uintptr_t)b.p;
  return x < y ? y - x < a.bytes : x - y < b.bytes;
}

// any of `a` with any of `b`
inline bool any_overlap(std::initializer_list<Span> a, std::initializer_list<Span> b) {
  for (const Span& x : a)
    for (const Span& y : b)
      if (overlap(x, y)) return true;
  return false;
}

// any two of `a`
inline bool any_overlap(std::initializer_list<Span> a) {
  for (const Span* x = a.begin(); x != a.end(); ++x)
    for (const Span* y = x + 1; y != a.end(); ++y)
      if (overlap(*x, *y)) return true;
  return false;
}

}  // namespace mla
