// Runs one scenario of device-to-host copies on the fake runtime
// (fake_hip/hip/hip_runtime.h); exits with 0 where it went as it should.
#include "../refrakt_amd/csrc/rf_stage.cpp"

#include <stdio.h>

#include <string>

static int fail(const char* what, size_t n) {
  printf("%s at %zu bytes\n", what, n);
  return 1;
}

static int copies(FakeStream s, size_t n) {
  std::vector<unsigned char> src(n), dst(n, 0);
  for (size_t i = 0; i < n; ++i) src[i] = (unsigned char)(i * 2654435761u >> 13);
  if (rfh::download(dst.data(), src.data(), n, &s) != hipSuccess) return fail("error", n);
  if (src != dst) return fail("wrong bytes", n);
  return 0;
}

// The stream's device is not the calling thread's.
static int other_device() {
  rfh::stage_hold();
  for (const size_t n : {(size_t)1 << 10, (size_t)1 << 20, (size_t)5 << 20, ((size_t)40 << 20) + 3}) {
    for (const int current : {0, 1, 0})
      for (const int stream : {1, 0}) {
        fake::device = current;
        if (int rc = copies(FakeStream{stream}, n)) return rc;
        if (fake::device != current) return fail("current device changed", n);
      }
  }
  rfh::stage_release();
  return fake::live_events || !fake::pinned.empty() ? fail("left over", 0) : 0;
}

// Staging that fails on its way is not the caller's error.
static int failing_stage() {
  rfh::stage_hold();
  const size_t n = ((size_t)40 << 20) + 3;
  for (const int records : {0, 1, 5}) {
    fake::records_left = records;
    if (int rc = copies(FakeStream{0}, n)) return rc;
    fake::records_left = -1;
    if (int rc = copies(FakeStream{0}, n)) return rc;
  }
  rfh::stage_release();
  return fake::live_events || !fake::pinned.empty() ? fail("left over", 0) : 0;
}

// A destination that the runtime knows is not written by the host: one
// transfer straight into it.
static int known_destination(hipMemoryType type, bool straight) {
  rfh::stage_hold();
  const size_t n = (size_t)5 << 20;
  std::vector<unsigned char> src(n, 7), dst(n, 0);
  FakeStream s{0};
  fake::known = dst.data();
  fake::known_type = type;
  if (rfh::download(dst.data(), src.data(), n, &s) != hipSuccess) return fail("error", n);
  if (src != dst) return fail("wrong bytes", n);
  if ((fake::last.dst == dst.data() && fake::last.n == n) != straight) return fail("other way", n);
  rfh::stage_release();
  return 0;
}

// More threads than stages: no stage is made for one copy.
static int many_threads() {
  rfh::stage_hold();
  fake::meet = 6;
  std::vector<int> rc(6, 0);
  std::vector<std::thread> ts;
  for (int t = 0; t < 6; ++t)
    ts.emplace_back([&rc, t] { rc[t] = copies(FakeStream{0}, ((size_t)5 << 20) + t); });
  for (auto& t : ts) t.join();
  for (int r : rc)
    if (r) return r;
  // two stages of two allocations each
  if (fake::pinned_peak > 4) return fail("too many stages", 5u << 20);
  // both idle, and for another device one of them gives way
  const size_t n = (size_t)5 << 20;
  if (int r = copies(FakeStream{1}, n)) return r;
  if (fake::last.n == n) return fail("not staged", n);
  if (fake::pinned_peak > 4) return fail("a third stage", n);
  rfh::stage_release();
  return fake::live_events || !fake::pinned.empty() ? fail("left over", 0) : 0;
}

int main(int argc, char** argv) {
  const std::string which = argc > 1 ? argv[1] : "";
  if (which == "other_device") return other_device();
  if (which == "failing_stage") return failing_stage();
  if (which == "many_threads") return many_threads();
  if (which == "pinned") return known_destination(hipMemoryTypeHost, true);
  if (which == "device") return known_destination(hipMemoryTypeDevice, true);
  if (which == "managed") return known_destination(hipMemoryTypeManaged, true);
  if (which == "unregistered") return known_destination(hipMemoryTypeUnregistered, false);
  return 2;
}
