// Second streams for the drivers that run two independent parts of one call side by side:
//  - launch_lu_large, launch_pf_large: the two halves of a batch, one half's panels (one
//    latency-bound workgroup per matrix) beside the other's trailing update;
//  - launch_tri_inverse: the two triangular factors' levels of a small batch;
//  - the float64 / complex slogpf gradients: the Parlett-Reid beside the LU.
//
// A device has up to SIDE_SLOTS side streams, each created when a caller stream first needs one
// more, with hipStreamNonBlocking (no implicit ordering with the null stream; every
// dependency is an explicit event) at the default priority, and kept, with its two events,
// until the process ends. A call takes the slot that its own stream used last, else a fresh
// one, else the one unused for longest, and holds it from its construction to its
// destructor, so that no two host threads record the same events. So callers on up to
// SIDE_SLOTS streams never queue behind each other's side work, and no call waits for
// another host thread: with every slot held, or under graph capture, it runs unsplit (the
// same bits).
#include <atomic>
#include <mutex>

#include "fermix_internal.h"

namespace fx {
namespace {

constexpr int SIDE_MAXDEV = 64;
constexpr int SIDE_SLOTS = 4;

}  // namespace

struct SideSlot {
  bool tried = false, ok = false, held = false;
  hipStream_t owner = nullptr;  // the caller stream that used it last (tried only)
  unsigned long long used = 0;  // when
  hipStream_t s2 = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};

namespace {

struct SidePool {
  std::mutex mu;
  unsigned long long clock = 0;
  SideSlot slot[SIDE_SLOTS];
};

SidePool g_side[SIDE_MAXDEV];

// The slot for s, marked as held, or nullptr.
SideSlot* take_slot(SidePool& p, hipStream_t s) {
  std::lock_guard<std::mutex> lk(p.mu);
  SideSlot *own = nullptr, *fresh = nullptr, *oldest = nullptr;
  for (SideSlot& t : p.slot) {
    if (t.held) continue;
    if (!t.tried) {
      if (!fresh) fresh = &t;
    } else if (t.ok) {
      if (t.owner == s) own = &t;
      if (!oldest || t.used < oldest->used) oldest = &t;
    }
  }
  if (!own && fresh) {
    fresh->tried = true;
    fresh->ok = hipStreamCreateWithFlags(&fresh->s2, hipStreamNonBlocking) == hipSuccess &&
                hipEventCreateWithFlags(&fresh->fork, hipEventDisableTiming) == hipSuccess &&
                hipEventCreateWithFlags(&fresh->join, hipEventDisableTiming) == hipSuccess;
    if (!fresh->ok) fresh = nullptr;
  }
  SideSlot* t = own ? own : fresh ? fresh : oldest;
  if (!t) return nullptr;
  t->held = true;
  t->owner = s;
  t->used = ++p.clock;
  return t;
}

}  // namespace

SideStream::SideStream(hipStream_t s, bool want) : s_(s) {
  if (!want) return;
  if (hipGetDevice(&dev_) != hipSuccess || dev_ < 0 || dev_ >= SIDE_MAXDEV) return;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return;
  slot_ = take_slot(g_side[dev_], s);
}

hipStream_t SideStream::side() const { return slot_ ? slot_->s2 : s_; }

int SideStream::fork() {
  if (!slot_ || forked_) return FX_ERR_LAUNCH;
  if (hipEventRecord(slot_->fork, s_) != hipSuccess || hipStreamWaitEvent(slot_->s2, slot_->fork, 0) != hipSuccess)
    return FX_ERR_LAUNCH;
  forked_ = true;
  return FX_OK;
}

int SideStream::join() {
  if (!forked_) return FX_OK;
  forked_ = false;
  if (hipEventRecord(slot_->join, slot_->s2) != hipSuccess || hipStreamWaitEvent(s_, slot_->join, 0) != hipSuccess)
    return FX_ERR_LAUNCH;
  return FX_OK;
}

SideStream::~SideStream() {
  join();
  if (!slot_) return;
  std::lock_guard<std::mutex> lk(g_side[dev_].mu);
  slot_->held = false;
}

int device_cus() {
  static std::atomic<int> cache[SIDE_MAXDEV];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SIDE_MAXDEV) return 256;
  int c = cache[dev].load(std::memory_order_relaxed);
  if (c > 0) return c;
  if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0) return 256;
  cache[dev].store(c, std::memory_order_relaxed);
  return c;
}

}  // namespace fx
