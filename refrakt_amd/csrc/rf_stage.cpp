// Device-to-host copies through pinned slots.
//
// hipMemcpy into pageable memory runs at 9 GB/s when the destination is fresh
// (its pages fault in on the one thread that copies) and at 18 GB/s when it is
// not; into pinned memory the same copy runs at 56 GB/s.  Here the device
// fills a ring of pinned slots and a few threads carry the slots to the
// destination, so page faults and host copies of one slot overlap the transfer
// of the next.  Into fresh memory, before and after: 1.2 MB 100 and 72 us,
// 4.2 MB 380 and 179 us, 33 MB 2.61 and 0.85 ms, 530 MB 50.3 and 13.1 ms.
#include "rf_stage.hpp"

#include <string.h>

#include <algorithm>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace rfh {
namespace {

constexpr size_t kDirect = 64 << 10;   // below this a plain copy is as fast
constexpr size_t kSlot = 4 << 20, kPiece = 512 << 10;
constexpr int kSlots = 8, kThreads = 8;
constexpr int kInFlight = 3;           // transfers queued before the oldest is waited for
constexpr int kPieces = (int)(kSlot / kPiece);

// Bytes per transfer: whole slots once the copy has many of them (a transfer
// costs about 12 us beside its bytes), half slots below, where the first
// transfer's time is not overlapped.
size_t chunk_bytes(size_t n) { return n >= 4 * kSlot ? kSlot : kSlot / 2; }

// One set of slots, used by one copy at a time.
class Stage {
 public:
  explicit Stage(int device) : device_(device) {}
  ~Stage() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
    }
    work_.notify_all();
    for (auto& t : threads_) t.join();
    for (hipEvent_t e : ev_)
      if (e) (void)hipEventDestroy(e);
    if (first_) (void)hipHostFree(first_);
    if (others_) (void)hipHostFree(others_);
  }
  Stage(const Stage&) = delete;
  Stage& operator=(const Stage&) = delete;

  int device() const { return device_; }

  // Slot 0 or, for many transfers, all slots (one allocation: each takes about
  // a millisecond) and the threads.
  bool ready(bool many) {
    auto pinned = [](void*& p, size_t bytes) {
      if (!p && hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess) p = nullptr;
      return p != nullptr;
    };
    if (!pinned(first_, kSlot) || (many && !pinned(others_, (kSlots - 1) * kSlot))) return false;
    slot_[0] = (char*)first_;
    for (int k = 1; many && k < kSlots; ++k) slot_[k] = (char*)others_ + (size_t)(k - 1) * kSlot;
    for (int k = 0; k < (many ? kSlots : 1); ++k)
      if (!ev_[k] && hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming) != hipSuccess) {
        ev_[k] = nullptr;
        return false;
      }
    if (many && threads_.empty()) {
      try {
        threads_.reserve(kThreads);
        for (int k = 0; k < kThreads; ++k) threads_.emplace_back([this] { run(); });
      } catch (...) {
        if (threads_.empty()) return false;  // fewer threads are enough
      }
    }
    return true;
  }

  hipError_t copy(char* host, const char* device, size_t n, hipStream_t s) {
    const size_t chunk = chunk_bytes(n), chunks = (n + chunk - 1) / chunk;
    if (chunks == 1) {
      hipError_t e = hipMemcpyAsync(slot_[0], device, n, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      if (e == hipSuccess) memcpy(host, slot_[0], n);
      return e;
    }
    hipError_t e = hipSuccess;
    size_t issued = 0, handed = 0;
    auto len = [&](size_t c) { return std::min(chunk, n - c * chunk); };
    while (handed < chunks && e == hipSuccess) {
      while (issued < chunks && issued - handed < (size_t)kInFlight && e == hipSuccess) {
        const int k = (int)(issued % kSlots);
        wait_slot(k);  // its last contents have been carried away
        e = hipMemcpyAsync(slot_[k], device + issued * chunk, len(issued), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev_[k], s);
        if (e == hipSuccess) ++issued;
      }
      if (e != hipSuccess) break;
      const int k = (int)(handed % kSlots);
      e = hipEventSynchronize(ev_[k]);
      if (e != hipSuccess) break;
      hand(k, host + handed * chunk, len(handed));
      ++handed;
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no transfer is left writing to a slot
    for (int k = 0; k < kSlots; ++k) wait_slot(k);
    return e;
  }

 private:
  struct Piece {
    char* dst;
    const char* src;
    size_t n;
    int slot;
  };

  // Queues slot k's n bytes in pieces.
  void hand(int k, char* dst, size_t n) {
    const int pieces = (int)((n + kPiece - 1) / kPiece);
    {
      std::lock_guard<std::mutex> lk(mu_);
      left_[k] = pieces;
      for (int p = 0; p < pieces; ++p) {
        const size_t o = (size_t)p * kPiece;
        queue_[(head_ + count_++) % kQueue] = Piece{dst + o, slot_[k] + o, std::min(kPiece, n - o), k};
      }
    }
    work_.notify_all();
  }

  void wait_slot(int k) {
    std::unique_lock<std::mutex> lk(mu_);
    done_.wait(lk, [&] { return left_[k] == 0; });
  }

  void run() {
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
      work_.wait(lk, [&] { return stop_ || count_ > 0; });
      if (count_ == 0) return;
      const Piece p = queue_[head_];
      head_ = (head_ + 1) % kQueue;
      --count_;
      lk.unlock();
      memcpy(p.dst, p.src, p.n);
      lk.lock();
      if (--left_[p.slot] == 0) done_.notify_all();
    }
  }

  static constexpr int kQueue = kSlots * kPieces;  // every piece of every slot
  int device_;
  void* first_ = nullptr;   // slot 0
  void* others_ = nullptr;  // the other slots
  char* slot_[kSlots] = {nullptr};
  hipEvent_t ev_[kSlots] = {nullptr};
  std::vector<std::thread> threads_;
  std::mutex mu_;
  std::condition_variable work_, done_;
  Piece queue_[kQueue];
  int head_ = 0, count_ = 0;
  int left_[kSlots] = {0};
  bool stop_ = false;
};

// The process' stages; copies of several threads take one each.  A copy that
// finds them taken is a plain one: a stage made for it (28 MB to pin, eight
// threads to start) costs more than it saves (eight threads with images of
// 4 MB: 1.0 to 1.5 ms a round, 0.7 to 0.85 so, 0.66 to 0.77 all plain).
struct Pool {
  std::mutex mu;
  int holders = 0;
  size_t made = 0;  // idle or in use
  std::vector<std::unique_ptr<Stage>> idle;
};
constexpr size_t kStages = 2;
Pool& pool() {
  static Pool* p = new Pool;  // outlives the runtime's teardown; emptied by the last stage_release
  return *p;
}

// A stage for the device, or null where all are in use.
std::unique_ptr<Stage> take(int device) {
  Pool& p = pool();
  std::unique_ptr<Stage> other;  // an idle stage of another device that gives way, freed here
  {
    std::lock_guard<std::mutex> lk(p.mu);
    for (size_t k = 0; k < p.idle.size(); ++k)
      if (p.idle[k]->device() == device) {
        std::unique_ptr<Stage> s = std::move(p.idle[k]);
        p.idle.erase(p.idle.begin() + (ptrdiff_t)k);
        return s;
      }
    p.idle.reserve(kStages);  // give does not allocate
    if (p.made < kStages) {
      ++p.made;
    } else if (!p.idle.empty()) {
      other = std::move(p.idle.back());
      p.idle.pop_back();
    } else {
      return nullptr;
    }
  }
  other.reset();
  try {
    return std::unique_ptr<Stage>(new Stage(device));
  } catch (...) {
    std::lock_guard<std::mutex> lk(p.mu);
    --p.made;
    throw;
  }
}

// Takes a stage back; it is kept where `good` and while contexts are there.
void give(std::unique_ptr<Stage> s, bool good) {
  Pool& p = pool();
  std::lock_guard<std::mutex> lk(p.mu);
  if (good && p.holders > 0) p.idle.push_back(std::move(s));
  else --p.made;
}  // else freed

// Makes a device current for its lifetime: events and pinned memory belong to
// the current device, and a slot's event is recorded on the copy's stream.
class OnDevice {
 public:
  explicit OnDevice(int device) {
    if (hipGetDevice(&before_) != hipSuccess) before_ = device;
    if (before_ != device) (void)hipSetDevice(device);
    device_ = device;
  }
  ~OnDevice() {
    if (before_ != device_) (void)hipSetDevice(before_);
  }
  OnDevice(const OnDevice&) = delete;
  OnDevice& operator=(const OnDevice&) = delete;

 private:
  int before_ = 0, device_ = 0;
};

hipError_t plain(void* host, const void* device, size_t n, hipStream_t s) {
  const hipError_t e = hipMemcpyAsync(host, device, n, hipMemcpyDeviceToHost, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace

hipError_t download(void* host, const void* device, size_t n, hipStream_t s) {
  if (n < kDirect) return plain(host, device, n, s);
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, host) == hipSuccess && at.type != hipMemoryTypeUnregistered)
    return plain(host, device, n, s);  // pinned (one transfer at full rate), or not the host's to write
  (void)hipGetLastError();             // not a pointer the runtime knows: the usual case
  hipDevice_t dev = 0;
  if (hipStreamGetDevice(s, &dev) != hipSuccess) {
    (void)hipGetLastError();
    return plain(host, device, n, s);
  }
  try {
    const OnDevice on(dev);
    if (std::unique_ptr<Stage> st = take(dev)) {
      const bool good = st->ready(n > chunk_bytes(n)) &&
                        st->copy((char*)host, (const char*)device, n, s) == hipSuccess;
      give(std::move(st), good);
      if (good) return hipSuccess;
      (void)hipGetLastError();  // of the stage, which is gone; the copy's own error shows again
    }
  } catch (...) {  // out of host memory before or after the copy, never during it
  }
  return plain(host, device, n, s);
}

void stage_hold() {
  Pool& p = pool();
  std::lock_guard<std::mutex> lk(p.mu);
  ++p.holders;
}

void stage_release() {
  std::vector<std::unique_ptr<Stage>> out;
  Pool& p = pool();
  std::lock_guard<std::mutex> lk(p.mu);
  if (--p.holders != 0) return;
  p.made -= p.idle.size();
  out.swap(p.idle);
}

}  // namespace rfh
