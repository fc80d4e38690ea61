// transfer.hpp -- a state between the device (tile order, FP64 or FP32) and
// the caller's array (reference order, FP64).
//
// The state moves in pieces through pinned host buffers: several host threads
// take pieces in turn, and each has the DMA of its next piece in flight while
// it permutes and converts the present one; a state of one piece takes one
// copy and one wait.  One pageable copy of the whole
// state and one thread's loop over its elements, into pages that the caller
// had not touched yet, moved 3 to 5 GB/s of the caller's array.  Reading the
// 512^2 vortex's 210 MB: FP32 45 -> 4.4 ms, FP64 72 -> 7.4; the 128^2 one's
// 13 MB: 1.45 -> 0.7 and 2.0 -> 0.8; setting it: 0.5 -> 0.4, 1.0 -> 0.6.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

namespace mxm {

// Pinned buffers of one piece each, shared by every solver and batch of the
// process: a transfer takes what it needs and gives it back when it ends.  At
// most kKept are kept for the next one, and none once the last object that
// may use them is gone.  Pinning memory takes 0.1 to 1 ms at first, which a
// buffer per object paid for each of them (and held for its life).
class PinnedPool {
 public:
  static constexpr size_t kPiece = 1 << 20;  // bytes of device state per piece
  static constexpr int kKept = 16;
  static PinnedPool &get() {
    static PinnedPool *pool = new PinnedPool;  // outlives every static object
    return *pool;
  }
  // nullptr where no pinned memory can be had
  char *take() {
    {
      std::lock_guard<std::mutex> l(m_);
      if (n_ > 0) return free_[--n_];
    }
    char *p = nullptr;
    if (hipHostMalloc(reinterpret_cast<void **>(&p), kPiece) == hipSuccess) return p;
    (void)hipGetLastError();  // handled by the caller, not the next launch's error
    return nullptr;
  }
  void give(char *p) {
    {
      std::lock_guard<std::mutex> l(m_);
      if (users_ > 0 && n_ < kKept) {
        free_[n_++] = p;
        return;
      }
    }
    (void)hipHostFree(p);
  }
  void join() {
    std::lock_guard<std::mutex> l(m_);
    ++users_;
  }
  void leave() {
    std::lock_guard<std::mutex> l(m_);
    if (--users_ > 0) return;
    while (n_ > 0) (void)hipHostFree(free_[--n_]);
  }

 private:
  PinnedPool() = default;
  std::mutex m_;
  char *free_[kKept] = {};
  int n_ = 0, users_ = 0;
};

// One buffer of the pool while it is used; pageable where the pool has none
// (copies then wait), empty where there is no memory at all.
struct PinnedPiece {
  char *p = PinnedPool::get().take();
  bool pinned = p != nullptr;
  PinnedPiece() {
    if (!pinned) p = static_cast<char *>(std::malloc(PinnedPool::kPiece));
  }
  PinnedPiece(const PinnedPiece &) = delete;
  PinnedPiece &operator=(const PinnedPiece &) = delete;
  ~PinnedPiece() {
    if (pinned)
      PinnedPool::get().give(p);
    else
      std::free(p);
  }
};

// What the transfers of one solver or batch keep between them.
struct HostPieces {
  static constexpr size_t kPiece = PinnedPool::kPiece;
  static constexpr int kThreads = 8;  // at most; each has two pieces
  hipEvent_t ev[2 * kThreads] = {};
  HostPieces() { PinnedPool::get().join(); }
  HostPieces(const HostPieces &) = delete;
  HostPieces &operator=(const HostPieces &) = delete;
  ~HostPieces() {
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
    PinnedPool::get().leave();
  }
  hipError_t events(int n) {
    for (int k = 0; k < n; ++k) {
      if (ev[k]) continue;
      const hipError_t e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
      if (e != hipSuccess) {
        ev[k] = nullptr;
        return e;
      }
    }
    return hipSuccess;
  }
};

// The device of a stream made current while its events are created: an event
// belongs to the device that was current, and is recorded only on that
// device's streams.
struct OnDevice {
  int before = -1, now;
  explicit OnDevice(int device) : now(device) {
    if (hipGetDevice(&before) != hipSuccess || before == now || hipSetDevice(now) != hipSuccess) before = now;
  }
  OnDevice(const OnDevice &) = delete;
  ~OnDevice() {
    if (before != now) (void)hipSetDevice(before);
  }
};

// Slots [0, slots) of `dev` (node values each) <-> elements ref_of[slot] of h
// (ref_of < 0: padding, zero on the device).  Returns when the caller may
// use h (TO_HOST) or drop it, with the stream idle.
template <bool TO_HOST, class R, class H>
hipError_t move_state(HostPieces &hp, R *dev, const int32_t *ref_of, int slots, size_t node, H *h, int device,
                      hipStream_t stream) {
  const int per = std::max<int>(1, (int)(HostPieces::kPiece / (node * sizeof(R))));  // slots per piece
  if ((size_t)per * node * sizeof(R) > HostPieces::kPiece) return hipErrorInvalidValue;
  const int pieces = (slots + per - 1) / per;
  if (pieces == 0) return hipStreamSynchronize(stream);
  // slots [begin, begin + n) between a piece and the caller's array
  auto elements = [&](int begin, int n, R *b) {
    for (int k = 0; k < n; ++k) {
      const int el = ref_of[begin + k];
      R *d = b + (size_t)k * node;
      if (el < 0) {
        if (!TO_HOST) std::fill(d, d + node, R(0));
        continue;
      }
      auto *u = h + (size_t)el * node;
      for (size_t v = 0; v < node; ++v) {
        if constexpr (TO_HOST)
          u[v] = double(d[v]);
        else
          d[v] = R(u[v]);
      }
    }
  };
  auto copy = [&](R *b, int begin, int n) {
    R *const d = dev + (size_t)begin * node;
    const size_t bytes = (size_t)n * node * sizeof(R);
    return TO_HOST ? hipMemcpyAsync(b, d, bytes, hipMemcpyDeviceToHost, stream)
                   : hipMemcpyAsync(d, b, bytes, hipMemcpyHostToDevice, stream);
  };
  if (pieces == 1) {  // nothing to overlap: one copy and one wait
    const PinnedPiece piece;
    if (!piece.p) return hipErrorOutOfMemory;
    R *const b = reinterpret_cast<R *>(piece.p);
    if (!TO_HOST) elements(0, slots, b);
    const hipError_t c = copy(b, 0, slots), w = hipStreamSynchronize(stream);
    if (c != hipSuccess || w != hipSuccess) return c != hipSuccess ? c : w;
    if (TO_HOST) elements(0, slots, b);
    return hipSuccess;
  }
  // a thread pays from about two pieces on
  const int threads = std::max(1, std::min({HostPieces::kThreads, pieces / 2, (int)std::thread::hardware_concurrency()}));
  const int ring = pieces > threads ? 2 : 1;  // pieces each thread has under way
  const OnDevice on(device);
  hipError_t e = hp.events(threads * ring);
  if (e != hipSuccess) return e;
  const std::vector<PinnedPiece> buffers(threads * ring);
  for (const PinnedPiece &b : buffers)
    if (!b.p) return hipErrorOutOfMemory;
  std::atomic<int> next{0}, error{(int)hipSuccess};
  auto work = [&](int t) {
    auto ok = [&](hipError_t r) {
      if (r != hipSuccess) error = (int)r;
      return r == hipSuccess && error == (int)hipSuccess;
    };
    if (t > 0 && !ok(hipSetDevice(device))) return;
    auto begin = [&](int c) { return c * per; };
    auto count = [&](int c) { return std::min(per, slots - c * per); };
    auto buf = [&](int s) { return reinterpret_cast<R *>(buffers[t * ring + s].p); };
    int piece[2] = {-1, -1};
    // the buffers in turn: wait for what is under way in one, finish it, put
    // the next piece under way
    bool more = true;
    for (int s = 0, idle = 0; idle < ring; s = ring == 2 ? 1 - s : 0) {
      const int at = t * ring + s;
      if (piece[s] >= 0) {
        if (!ok(hipEventSynchronize(hp.ev[at]))) return;
        if (TO_HOST) elements(begin(piece[s]), count(piece[s]), buf(s));
        piece[s] = -1;
      }
      int c = more ? next.fetch_add(1) : pieces;
      if (c >= pieces) {
        more = false;
        ++idle;
        continue;
      }
      idle = 0;
      if (!TO_HOST) elements(begin(c), count(c), buf(s));
      if (!ok(copy(buf(s), begin(c), count(c))) || !ok(hipEventRecord(hp.ev[at], stream))) return;
      piece[s] = c;
    }
  };
  std::vector<std::thread> pool;
  pool.reserve(threads);
  for (int t = 1; t < threads; ++t) {
    try {
      pool.emplace_back(work, t);
    } catch (...) {
      break;  // the threads there are do the work
    }
  }
  work(0);
  for (auto &t : pool) t.join();
  e = hipStreamSynchronize(stream);  // also after an error: nothing under way touches h or the buffers
  return error != (int)hipSuccess ? (hipError_t)error.load() : e;
}

}  // namespace mxm
