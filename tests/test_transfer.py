"""State transfers between the device and the caller (csrc/transfer.hpp),
compiled for the host against a small stand-in for the HIP calls they make: a
stream that runs its copies later on a thread of its own, with the calls that
can fail made to fail.  Every piece count (none, one, a few, many, ragged last
pieces), both directions, both state types, padding slots."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIP = r"""
#pragma once
#include <atomic>
#include <condition_variable>
#include <chrono>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipEventDisableTiming = 2;
struct Stream {
  int device;
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  long put = 0, done = 0;
  bool stop = false;
  std::thread t;
  explicit Stream(int d) : device(d), t([this] { run(); }) {}
  ~Stream() {
    { std::lock_guard<std::mutex> l(m); stop = true; }
    cv.notify_all();
    t.join();
  }
  void run() {
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      cv.wait(l, [&] { return stop || !q.empty(); });
      if (q.empty()) return;
      auto f = std::move(q.front());
      q.pop_front();
      l.unlock();
      std::this_thread::sleep_for(std::chrono::microseconds(50));
      f();
      l.lock();
      ++done;
      cv.notify_all();
    }
  }
  long add(std::function<void()> f) {
    std::lock_guard<std::mutex> l(m);
    q.push_back(std::move(f));
    cv.notify_all();
    return ++put;
  }
  long last() { std::lock_guard<std::mutex> l(m); return put; }
  void wait(long n) {
    std::unique_lock<std::mutex> l(m);
    cv.wait(l, [&] { return done >= n; });
  }
};
typedef Stream *hipStream_t;
struct Event { int device; Stream *s = nullptr; long at = 0; };
typedef Event *hipEvent_t;
inline thread_local int cur_device = 0;
inline hipError_t last_error = hipSuccess;
inline int fail_events = 0, fail_pinned = 0, fail_copy = 0, live_events = 0, made_pinned = 0;
inline std::atomic<int> live_pinned{0};
inline hipError_t bad(hipError_t e) { return last_error = e; }
inline hipError_t hipGetLastError() { auto e = last_error; last_error = hipSuccess; return e; }
inline hipError_t hipGetDevice(int *d) { *d = cur_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { cur_device = d; return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n) {
  if (fail_pinned > 0) { --fail_pinned; return bad(hipErrorOutOfMemory); }
  ++live_pinned, ++made_pinned;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) { --live_pinned; std::free(p); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  if (fail_events > 0 && --fail_events == 0) return bad(hipErrorOutOfMemory);
  ++live_events;
  *e = new Event{cur_device};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { --live_events; delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (!e || e->device != s->device) return bad(hipErrorInvalidHandle);
  e->s = s, e->at = s->last();
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (!e) return bad(hipErrorInvalidHandle);
  if (e->s) e->s->wait(e->at);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { s->wait(s->last()); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  if (fail_copy > 0 && --fail_copy == 0) return bad(hipErrorInvalidValue);
  st->add([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
"""

MAIN = r"""
#include "transfer.hpp"

#include <cstdio>

using namespace mxm;

#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

// elements 0 .. n-1 in mixed order over slots, every fifth slot padding
static std::vector<int32_t> order(int slots, int &n) {
  std::vector<int32_t> r(slots, -1);
  n = 0;
  for (int s = 0; s < slots; ++s)
    if (s % 5 != 3) r[s] = n++;
  for (int s = 0; s < slots; ++s)
    if (r[s] >= 0) r[s] = n - 1 - r[s];
  return r;
}

template <class R>
int both_ways(HostPieces &hp, int slots, size_t node, int device, Stream *st) {
  int n = 0;
  const auto ref = order(slots, n);
  std::vector<double> h(n * node), back(n * node, -7.0);
  for (size_t k = 0; k < h.size(); ++k) h[k] = 1.0 + 1e-9 * double(k * 2654435761u % 1000003);
  std::vector<R> dev(slots * node, R(-3));
  const double *in = h.data();
  CHECK(move_state<false>(hp, dev.data(), ref.data(), slots, node, in, device, st) == hipSuccess);
  for (int s = 0; s < slots; ++s)
    for (size_t v = 0; v < node; ++v)
      CHECK(dev[s * node + v] == (ref[s] < 0 ? R(0) : R(h[ref[s] * node + v])));
  CHECK(move_state<true>(hp, dev.data(), ref.data(), slots, node, back.data(), device, st) == hipSuccess);
  for (size_t k = 0; k < h.size(); ++k) CHECK(back[k] == double(R(h[k])));
  return 0;
}

template <class R>
int sizes(Stream &st) {
  HostPieces hp;
  for (size_t node : {1, 7, 50, 952}) {
    const int per = int(HostPieces::kPiece / (node * sizeof(R)));
    if (node == 1) {
      CHECK(!both_ways<R>(hp, 3 * per + 1, node, 0, &st));
      continue;
    }
    for (int slots : {0, 1, 24, per - 1, per, per + 1, 2 * per, 2 * per + 1, 3 * per, 4 * per + 3, 17 * per + 5, 40 * per - 1})
      CHECK(!both_ways<R>(hp, slots, node, 0, &st));
  }
  return 0;
}

int main(int argc, char **argv) {
  const std::string what = argv[1];
  Stream st(0);
  if (what == "sizes") return sizes<double>(st) || sizes<float>(st);
  if (what == "pool") {  // buffers are shared, bounded, and gone with the last object
    {
      HostPieces a;
      CHECK(!both_ways<float>(a, 24, 50, 0, &st));
      CHECK(made_pinned == 1 && live_events == 0);  // one piece: one buffer, no events
      {
        HostPieces b;
        CHECK(!both_ways<float>(b, 24, 50, 0, &st) && !both_ways<double>(a, 30, 50, 0, &st));
        CHECK(made_pinned == 1);
      }
      CHECK(!both_ways<double>(a, 60000, 50, 0, &st));
      CHECK(live_pinned <= PinnedPool::kKept);
      const int made = made_pinned;
      CHECK(!both_ways<double>(a, 60000, 50, 0, &st));
      CHECK(made_pinned == made);
      std::vector<PinnedPiece> many(3 * PinnedPool::kKept);
      CHECK(live_pinned == 3 * PinnedPool::kKept);
      many.clear();
      CHECK(live_pinned == PinnedPool::kKept);
    }
    CHECK(live_pinned == 0 && live_events == 0);
    // several objects, streams and threads at once
    std::vector<std::thread> t;
    std::atomic<int> bad{0};
    for (int k = 0; k < 6; ++k)
      t.emplace_back([&bad, k] {
        Stream mine(0);
        HostPieces hp;
        for (int r = 0; r < 4; ++r) bad += both_ways<float>(hp, 3000 * (k + 1) + r, 50, 0, &mine);
      });
    for (auto &x : t) x.join();
    CHECK(!bad && live_pinned == 0);
  }
  if (what == "events") {  // a call that could not get its events fails; the next one works
    for (int k = 1; k <= 3; ++k) {
      HostPieces hp;
      std::vector<float> dev(400000 * 4);
      std::vector<int32_t> ref(400000, -1);
      std::vector<double> h(4);
      const double *in = h.data();
      fail_events = k;
      CHECK(move_state<false>(hp, dev.data(), ref.data(), 400000, size_t(4), in, 0, &st) != hipSuccess);
      fail_events = 0;
      CHECK(!both_ways<float>(hp, 400000, 4, 0, &st));
    }
    CHECK(live_events == 0 && live_pinned == 0);
  }
  if (what == "pinned") {  // no pinned memory: pageable, and no error left behind
    HostPieces hp;
    fail_pinned = 1 << 20;
    CHECK(!both_ways<double>(hp, 24, 50, 0, &st));
    CHECK(!both_ways<double>(hp, 30000, 50, 0, &st));
    CHECK(hipGetLastError() == hipSuccess);
    fail_pinned = 0;
    CHECK(!both_ways<double>(hp, 60000, 50, 0, &st));
  }
  if (what == "device") {  // another device is current
    HostPieces hp;
    hipSetDevice(3);
    CHECK(!both_ways<double>(hp, 60000, 50, 0, &st));
    int d = -1;
    hipGetDevice(&d);
    CHECK(d == 3);
  }
  if (what == "copy") {  // a copy that fails: the call reports it, with nothing under way
    for (int k = 1; k < 40; k += 3) {
      HostPieces hp;
      int n = 0;
      const auto ref = order(60000, n);
      std::vector<double> dev(60000 * 50), h((size_t)n * 50);
      fail_copy = k;
      const hipError_t e = move_state<true>(hp, dev.data(), ref.data(), 60000, size_t(50), h.data(), 0, &st);
      CHECK((fail_copy > 0) == (e == hipSuccess));
      CHECK(st.done == st.put);
      fail_copy = 0;
    }
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("transfer")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(HIP)
    (d / "main.cpp").write_text("#include <string>\n" + MAIN)
    exe = str(d / "transfer")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", "-I", str(d), "-I",
                    os.path.join(ROOT, "mojoxm_amd", "csrc"), str(d / "main.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("what", ["sizes", "events", "pinned", "device", "pool", "copy"])
def test_transfer(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
