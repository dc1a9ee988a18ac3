// Buffers of constants that are made on their first use.
#pragma once
#include <stddef.h>

namespace rfh {

// Allocates n bytes for b and has fill(b.p) fill them, unless that is done.  A
// buffer that could not be filled is given back, so the next call tries again
// instead of reading what was never written.  Errors are an enum whose zero
// value is success.
template <class Buf, class Fill>
auto fill_once(Buf& b, size_t n, Fill fill) -> decltype(b.alloc(n)) {
  decltype(b.alloc(n)) e{};
  const auto ok = e;
  if (b.p) return ok;
  e = b.alloc(n);
  if (e == ok) e = fill(b.p);
  if (e != ok) b.release();
  return e;
}

}  // namespace rfh
