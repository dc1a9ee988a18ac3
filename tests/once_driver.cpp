// fill_once (rf_once.hpp) with a buffer and a fill that fail on request; exits
// with 0 where it went as it should.
#include "../refrakt_amd/csrc/rf_once.hpp"

#include <stdlib.h>

enum Error { kOk = 0, kBad = 7 };

struct Buf {
  void* p = nullptr;
  int allocs = 0, releases = 0;
  bool refuse = false;
  Error alloc(size_t n) {
    ++allocs;
    if (refuse) return kBad;
    p = malloc(n);
    return kOk;
  }
  void release() {
    ++releases;
    free(p);
    p = nullptr;
  }
};

int main() {
  Buf b;
  int fills = 0;
  Error next = kBad;
  auto fill = [&](void* p) {
    ++fills;
    return p == b.p ? next : kBad;
  };
  b.refuse = true;
  if (rfh::fill_once(b, 64, fill) != kBad || b.p || fills != 0) return 1;
  b.refuse = false;
  if (rfh::fill_once(b, 64, fill) != kBad || b.p || fills != 1) return 2;  // not kept half made
  next = kOk;
  if (rfh::fill_once(b, 64, fill) != kOk || !b.p || fills != 2) return 3;  // tried again
  if (rfh::fill_once(b, 64, fill) != kOk || fills != 2 || b.allocs != 3) return 4;  // once
  b.release();
  return 0;
}
