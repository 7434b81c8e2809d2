// Host code without HIP types: compiled into the library, and by itself in the CPU tests.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <deque>
#include <exception>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace fh {

// Workgroups of `threads` threads that a launch may have along x: HIP refuses gridDim.x blockDim.x >= 2^32.
inline int64_t max_workgroups(int threads) { return (((int64_t)1 << 32) - 1) / threads; }

// f(first, count) for `items` cut into launches of `each` workgroups an item
template <typename F>
void for_launches(int64_t items, int64_t each, int threads, F&& f) {
  const int64_t per = std::max<int64_t>(1, max_workgroups(threads) / each);
  for (int64_t i = 0; i < items; i += per) f(i, std::min(per, items - i));
}

// Timed spans on a stream: an event pair each, read back in the order in which the spans ended.  No more than kMax ended
// spans wait for that: the next one takes the older half first, which waits for their work, behind which that of the
// other half is queued, so that the device does not idle.  Within a call the events are used again, at most two for each
// waiting and each open span (the (T) of o = 64, v = 320 has 23 000 spans); flush() leaves none.
// Rt: Event, Stream and bool create(Event&), record(Event, Stream), wait(Event), elapsed(float& ms, Event, Event),
// void destroy(Event).
template <typename Rt>
class Spans {
 public:
  struct Span {
    std::string name;
    double flops = 0.0, bytes = 0.0;
    typename Rt::Event a{}, b{};
  };
  static constexpr size_t kMax = 32;
  Spans() = default;
  Spans(const Spans&) = delete;
  Spans& operator=(const Spans&) = delete;
  ~Spans() {
    for (Span& p : ended_) give(p);
    clear();
  }
  // false: no event could be had or recorded
  bool begin(Span& p, typename Rt::Stream s) {
    if (!take(p.a)) return false;
    if (!take(p.b)) {
      free_.push_back(p.a);
      return false;
    }
    if (Rt::record(p.a, s)) return true;
    give(p);
    return false;
  }
  template <typename F>
  void end(Span& p, typename Rt::Stream s, F&& sink) {
    if (!Rt::record(p.b, s)) {
      give(p);
      return;
    }
    ended_.push_back(p);
    if (ended_.size() > kMax) resolve(kMax / 2, sink);
  }
  // sink(span, ms) for all ended spans
  template <typename F>
  void flush(F&& sink) {
    resolve(ended_.size(), sink);
    clear();
  }

 private:
  // the n spans that ended first
  template <typename F>
  void resolve(size_t n, F&& sink) {
    for (; n > 0 && !ended_.empty(); --n) {
      Span p = ended_.front();
      ended_.pop_front();
      float ms = 0.f;
      if (Rt::wait(p.b) && Rt::elapsed(ms, p.a, p.b)) sink(p, ms);
      give(p);
    }
  }
  void clear() {
    for (auto e : free_) Rt::destroy(e);
    free_.clear();
  }
  bool take(typename Rt::Event& e) {
    if (free_.empty()) return Rt::create(e);
    e = free_.back();
    free_.pop_back();
    return true;
  }
  void give(Span& p) {
    free_.push_back(p.a);
    free_.push_back(p.b);
  }
  std::deque<Span> ended_;
  std::vector<typename Rt::Event> free_;
};

// What several users of a process lend one another: take() gives an idle one (of a device) or none, give() keeps at most
// kKeep of them idle, and the last user to leave frees those.
template <typename T>
class IdlePool {
 public:
  static constexpr size_t kKeep = 2;
  void enter() {
    std::lock_guard<std::mutex> g(m_);
    ++users_;
  }
  void leave() {
    std::vector<std::unique_ptr<T>> gone;
    std::lock_guard<std::mutex> g(m_);
    if (--users_ == 0) gone.swap(idle_);
  }
  std::unique_ptr<T> take(int device) {
    std::lock_guard<std::mutex> g(m_);
    for (auto& p : idle_)
      if (p->device == device) {
        std::swap(p, idle_.back());
        std::unique_ptr<T> r = std::move(idle_.back());
        idle_.pop_back();
        return r;
      }
    return nullptr;
  }
  void give(std::unique_ptr<T> p) {
    std::lock_guard<std::mutex> g(m_);
    if (users_ > 0 && idle_.size() < kKeep) idle_.push_back(std::move(p));
  }

 private:
  std::mutex m_;
  int users_ = 0;
  std::vector<std::unique_ptr<T>> idle_;
};

// Sizes from which a copy in chunks is the faster one, with the pinned buffers at hand. To the host 4 MiB: 4.5, 12, 24 MiB
// into one array 232, 460, 750 us against 277, 705, 1410, into new memory each time 310, 870, 1270 against 370, 1450,
// 2610. To the device 32 MiB: 6, 16, 24, 40 MiB from one array 273, 537, 745, 1150 us against 204, 481, 697, 1420,
// from new memory 318, 590, 800, 1250 against 245, 600, 895, 1480.
inline bool chunks_pay(size_t n, bool to_host) { return n >= (size_t)(to_host ? 4 : 32) << 20; }
// Whether to make the buffers, which takes a millisecond: when the copies that missed them, this one among them, would
// have gained as much (24 MiB to the host, five times that to the device).
inline bool chunks_worth_making(size_t& missed, size_t n, bool to_host) {
  missed += to_host ? n : n / 5;
  return missed >= (size_t)24 << 20;
}

// Copy of n bytes between the device and host memory in chunks of Rt::kChunk through pinned buffers, two a thread, chunk i
// by thread i mod Rt::kThreads: the DMA of a chunk runs while those before it are moved between the buffers and
// the host memory. false: a step failed; then too nothing is in flight any more.
// Rt: char* buf(t, k); bool enter() on a thread's first step, start(t, k, offset, bytes) and mark(t, k) a DMA, wait(t, k) for
// its mark; void drain() waits for everything started.
template <typename Rt>
bool copy_chunked(Rt& rt, char* host, size_t n, bool to_host) {
  constexpr size_t CH = Rt::kChunk;
  const size_t nch = (n + CH - 1) / CH;
  bool good[Rt::kThreads] = {};
  auto work = [&](int t) {
    if (!rt.enter()) return;
    auto len = [&](size_t i) { return std::min(CH, n - i * CH); };
    size_t in[2] = {nch, nch};   // chunk in flight in each buffer
    auto finish = [&](int k) {
      if (in[k] == nch) return true;
      if (!rt.wait(t, k)) return false;
      if (to_host) std::memcpy(host + in[k] * CH, rt.buf(t, k), len(in[k]));
      in[k] = nch;
      return true;
    };
    int k = 0;
    for (size_t i = t; i < nch; i += Rt::kThreads, k ^= 1) {
      if (!finish(k)) return;
      if (!to_host) std::memcpy(rt.buf(t, k), host + i * CH, len(i));
      if (!rt.start(t, k, i * CH, len(i)) || !rt.mark(t, k)) return;
      in[k] = i;
    }
    good[t] = finish(k) && finish(k ^ 1);
  };
  std::vector<std::thread> th;
  int started = 1;
  try {
    th.reserve(Rt::kThreads - 1);
    for (; started < Rt::kThreads; ++started) th.emplace_back(work, started);
  } catch (const std::exception&) {
    // no more threads: this one takes their chunks
  }
  work(0);
  for (int t = started; t < Rt::kThreads; ++t) work(t);
  for (auto& x : th) x.join();
  if (std::all_of(good, good + Rt::kThreads, [](bool g) { return g; })) return true;
  rt.drain();
  return false;
}

}  // namespace fh
