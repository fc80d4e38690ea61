// transfer.hpp -- a state between the device (tile order, FP64 or FP32) and
// the caller's array (reference order, FP64).
//
// The state moves in pieces through pinned host buffers: several host threads
// take pieces in turn, and each has the DMA of its next piece in flight while
// it permutes and converts the present one.  One pageable copy of the whole
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
#include <thread>
#include <vector>

namespace mxm {

// Pinned buffers of the transfers of one solver or batch, kept between them
// (pageable ones where no pinned memory can be had: the copies then wait).
struct HostPieces {
  static constexpr size_t kPiece = 1 << 20;  // bytes of device state per piece
  static constexpr int kThreads = 8;         // at most; each has two pieces
  char *p = nullptr;
  size_t size = 0;
  bool pinned = false;
  hipEvent_t ev[2 * kThreads] = {};
  HostPieces() = default;
  HostPieces(const HostPieces &) = delete;
  HostPieces &operator=(const HostPieces &) = delete;
  ~HostPieces() {
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
    release();
  }
  void release() {
    if (p && pinned)
      (void)hipHostFree(p);
    else
      std::free(p);
    p = nullptr, size = 0;
  }
  // n buffers, of `bytes` in all
  hipError_t reserve(int n, size_t bytes) {
    for (int k = 0; k < n; ++k) {
      if (ev[k]) continue;
      const hipError_t e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
      if (e != hipSuccess) {
        ev[k] = nullptr;
        return e;
      }
    }
    if (bytes <= size) return hipSuccess;
    bytes = std::max(bytes, std::min(2 * size, 2 * kThreads * kPiece));
    release();
    pinned = hipHostMalloc(reinterpret_cast<void **>(&p), bytes) == hipSuccess;
    if (!pinned) {
      (void)hipGetLastError();  // handled here, not the next launch's error
      p = static_cast<char *>(std::malloc(bytes));
      if (!p) return hipErrorOutOfMemory;
    }
    size = bytes;
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
  // a thread pays from about two pieces on
  const int threads = std::max(1, std::min({HostPieces::kThreads, pieces / 2, (int)std::thread::hardware_concurrency()}));
  const int ring = pieces > threads ? 2 : 1;  // pieces each thread has under way
  const OnDevice on(device);
  // a small state takes what it needs: pinning a whole piece for it cost its
  // first transfer 40 to 50 us (5^3 Euler, P = 2)
  const size_t stride = ((size_t)std::min(per, slots) * node * sizeof(R) + 255) / 256 * 256;
  hipError_t e = hp.reserve(threads * ring, (size_t)threads * ring * stride);
  if (e != hipSuccess) return e;
  std::atomic<int> next{0}, error{(int)hipSuccess};
  auto work = [&](int t) {
    auto ok = [&](hipError_t r) {
      if (r != hipSuccess) error = (int)r;
      return r == hipSuccess && error == (int)hipSuccess;
    };
    if (t > 0 && !ok(hipSetDevice(device))) return;
    auto begin = [&](int c) { return c * per; };
    auto count = [&](int c) { return std::min(per, slots - c * per); };
    auto buf = [&](int s) { return reinterpret_cast<R *>(hp.p + (size_t)(t * ring + s) * stride); };
    int piece[2] = {-1, -1};
    auto elements = [&](int c, R *b) {
      for (int k = 0; k < count(c); ++k) {
        const int el = ref_of[begin(c) + k];
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
    // the buffers in turn: wait for what is under way in one, finish it, put
    // the next piece under way
    bool more = true;
    for (int s = 0, idle = 0; idle < ring; s = ring == 2 ? 1 - s : 0) {
      const int at = t * ring + s;
      if (piece[s] >= 0) {
        if (!ok(hipEventSynchronize(hp.ev[at]))) return;
        if (TO_HOST) elements(piece[s], buf(s));
        piece[s] = -1;
      }
      int c = more ? next.fetch_add(1) : pieces;
      if (c >= pieces) {
        more = false;
        ++idle;
        continue;
      }
      idle = 0;
      if (!TO_HOST) elements(c, buf(s));
      R *d = dev + (size_t)begin(c) * node;
      const size_t bytes = (size_t)count(c) * node * sizeof(R);
      if (!ok(TO_HOST ? hipMemcpyAsync(buf(s), d, bytes, hipMemcpyDeviceToHost, stream)
                      : hipMemcpyAsync(d, buf(s), bytes, hipMemcpyHostToDevice, stream)) ||
          !ok(hipEventRecord(hp.ev[at], stream)))
        return;
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
