"""The library's host code without HIP types (csrc/fh_host.h), compiled by itself and run on the CPU."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fermi.jl_amd", "csrc")


def run_cpp(tmp_path, body):
    src, exe = str(tmp_path / "t.cpp"), str(tmp_path / "t")
    with open(src, "w") as f:
        f.write('#include "fh_host.h"\n#include <cstdio>\n#include <cstdlib>\n'
                '#define CHECK(x) do { if (!(x)) { printf("line %d: %s\\n", __LINE__, #x); exit(1); } } while (0)\n' + body)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", CSRC, src, "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    return r.stdout


def test_launches_below_the_grid_limit(tmp_path):
    """Every item in one launch, no launch of 2^32 threads: the (ss|ss) integrals of 181 and 251 uncontracted s functions
    (pairs of functions against as many kets, 64 a workgroup of 1024 threads), 2^31 items of one workgroup, few of many."""
    run_cpp(tmp_path, """
int main() {
  auto check = [](int64_t items, int64_t each, int threads, int64_t launches) {
    int64_t next = 0, n = 0;
    fh::for_launches(items, each, threads, [&](int64_t first, int64_t count) {
      CHECK(first == next && count > 0 && count * each * threads < (int64_t)1 << 32);
      next += count;
      ++n;
    });
    CHECK(next == items && n == launches);
  };
  for (int64_t n : {181, 251}) {
    const int64_t pairs = n * (n + 1) / 2;
    check(pairs, (pairs + 63) / 64, 1024, n == 181 ? 2 : 4);
  }
  check((int64_t)1 << 31, 1, 256, 129);
  check(5, 4000000, 1024, 5);
  check(1, 1, 64, 1);
  check(0, 1, 64, 0);
}
""")


def test_spans_hold_few_events(tmp_path):
    """A call of 5700 chunks with four spans each inside one: every span is read back once, with its own time, in the
    order of their ends; the events at hand stay below two for each of the spans that may wait and the open ones, and none
    is left. An event that cannot be made or recorded loses no other."""
    run_cpp(tmp_path, """
#include <map>
#include <set>
static std::set<int> live;
static size_t most = 0;
static int made = 0, clock_ = 0, fail_create = -1, fail_record = -1, records = 0, waits = 0;
static std::map<int, int> at;
struct Rt {
  using Event = int;
  using Stream = int;
  static bool create(int& e) {
    if (made == fail_create) return false;
    e = made++;
    live.insert(e);
    most = std::max(most, live.size());
    return true;
  }
  static void destroy(int e) { CHECK(live.erase(e) == 1); }
  static bool record(int e, int) {
    CHECK(live.count(e));
    if (records++ == fail_record) return false;
    at[e] = ++clock_;
    return true;
  }
  static bool wait(int e) { ++waits; return live.count(e) == 1; }
  static bool elapsed(float& ms, int a, int b) { ms = (float)(at[b] - at[a]); return true; }
};
using S = fh::Spans<Rt>;
int main() {
  {
    S spans;
    int seen = 0, inner = 0;
    auto sink = [&](const S::Span& p, float ms) {
      ++seen;
      if (p.name == "outer") CHECK(ms == 2 * 4 * 5700 + 1);
      else { CHECK(p.flops == inner++); CHECK(ms == 1); }
    };
    S::Span outer;
    outer.name = "outer";
    CHECK(spans.begin(outer, 0));
    for (int k = 0; k < 4 * 5700; ++k) {
      S::Span p;
      p.flops = k;
      CHECK(spans.begin(p, 0));
      spans.end(p, 0, sink);
      CHECK(k - inner <= (int)S::kMax);
      if (k < (int)S::kMax) CHECK(waits == 0);
    }
    spans.end(outer, 0, sink);
    CHECK(seen < 4 * 5700);
    spans.flush(sink);
    CHECK(seen == 4 * 5700 + 1);
    CHECK(most <= 2 * (S::kMax + 3) && live.empty());
    for (int k = 0; k < 3; ++k) {   // the next call; these are not flushed
      S::Span p;
      CHECK(spans.begin(p, 0));
      spans.end(p, 0, sink);
    }
    CHECK(live.size() == 6);
  }
  CHECK(live.empty());
  for (int f = 0; f < 6; ++f) {
    S spans;
    made = records = 0;
    fail_create = f < 2 ? f : -1;
    fail_record = f < 2 ? -1 : f - 2;
    int ok = 0, seen = 0;
    for (int k = 0; k < 3; ++k) {
      S::Span p;
      if (!spans.begin(p, 0)) { fail_create = fail_record = -1; continue; }
      ++ok;
      spans.end(p, 0, [](const S::Span&, float) {});
    }
    spans.flush([&](const S::Span&, float) { ++seen; });
    CHECK(ok == (f == 3 || f == 5 ? 3 : 2) && seen == 2);
  }
  CHECK(live.empty());
  return 0;
}
""")


def test_chunked_copy(tmp_path):
    """copy_chunked with DMAs that move their bytes as late as they may (at the wait for their mark, or at the drain): both
    directions, sizes around a chunk and a round of buffers; and with each step failing in turn, no chunk is in flight
    when it returns."""
    run_cpp(tmp_path, """
#include <mutex>
struct Rt {
  static constexpr int kThreads = 3;
  static constexpr size_t kChunk = 16;
  std::mutex m;
  char* dev;
  bool to_host;
  int fail, step = 0;
  struct Dma { size_t at = 0, n = 0; bool flying = false; } dma[kThreads][2];
  char pinned[kThreads][2][kChunk];
  Rt(char* d, bool h, int f) : dev(d), to_host(h), fail(f) {}
  bool good() { std::lock_guard<std::mutex> g(m); return step++ != fail; }
  void land(int t, int k) {
    Dma& d = dma[t][k];
    if (d.flying) {
      if (to_host) std::memcpy(pinned[t][k], dev + d.at, d.n);
      else std::memcpy(dev + d.at, pinned[t][k], d.n);
    }
    d.flying = false;
  }
  char* buf(int t, int k) { CHECK(!dma[t][k].flying); return pinned[t][k]; }
  bool enter() { return good(); }
  bool start(int t, int k, size_t at, size_t n) {
    CHECK(!dma[t][k].flying && n > 0 && n <= kChunk);
    if (!good()) return false;
    dma[t][k].at = at;
    dma[t][k].n = n;
    dma[t][k].flying = true;
    return true;
  }
  bool mark(int, int) { return good(); }
  bool wait(int t, int k) {
    if (!good()) return false;
    land(t, k);
    return true;
  }
  void drain() { for (int t = 0; t < kThreads; ++t) for (int k = 0; k < 2; ++k) land(t, k); }
};
int main() {
  for (bool to_host : {false, true})
    for (size_t n : {1, 15, 16, 17, 48, 95, 96, 97, 500})
      for (int fail = -1; ; ++fail) {
        std::vector<char> dev(n), host(n), want(n);
        for (size_t i = 0; i < n; ++i) want[i] = (char)(i * 7 + 1);
        (to_host ? dev : host) = want;
        Rt rt(dev.data(), to_host, fail);
        const bool ok = fh::copy_chunked(rt, host.data(), n, to_host);
        for (auto& t : rt.dma) for (auto& d : t) CHECK(!d.flying);
        if (ok) CHECK(host == want && dev == want);
        if (fail < 0) CHECK(ok);
        else if (rt.step > fail) CHECK(!ok);
        else break;
      }
}
""")


def test_chunked_copy_sizes(tmp_path):
    """Copies in chunks from 4 MiB to the host and from 32 MiB to the device on; the buffers are made for one copy of 24 or
    120 MiB or for several that come to as much."""
    run_cpp(tmp_path, """
int main() {
  const size_t M = (size_t)1 << 20;
  for (bool to_host : {false, true}) {
    const size_t from = (to_host ? 4 : 32) * M, once = (to_host ? 24 : 120) * M;
    CHECK(!fh::chunks_pay(from - 8, to_host) && fh::chunks_pay(from, to_host));
    size_t missed = 0;
    CHECK(!fh::chunks_worth_making(missed, once - 8, to_host));
    missed = 0;
    CHECK(fh::chunks_worth_making(missed, once, to_host) && fh::chunks_worth_making(missed, from, to_host));
  }
  size_t missed = 0;
  CHECK(!fh::chunks_worth_making(missed, 11 * M, true) && !fh::chunks_worth_making(missed, 40 * M, false));
  CHECK(fh::chunks_worth_making(missed, 5 * M, true));
}
""")


def test_idle_pool(tmp_path):
    """Lent objects: one user at a time, of the device asked for, no more than two idle, none after the last user left; from
    eight threads as from one."""
    run_cpp(tmp_path, """
#include <atomic>
static std::atomic<int> alive{0};
struct Thing {
  const int device;
  std::atomic<int> held{0};
  explicit Thing(int d) : device(d) { ++alive; }
  ~Thing() { --alive; }
};
int main() {
  fh::IdlePool<Thing> pool;
  pool.enter();
  CHECK(!pool.take(0));
  for (int d : {0, 1, 1}) pool.give(std::make_unique<Thing>(d));
  CHECK(alive == 2 && !pool.take(2));
  auto a = pool.take(1);
  CHECK(a && a->device == 1 && !pool.take(1));
  pool.give(std::move(a));
  pool.enter();
  pool.leave();
  CHECK(alive == 2);
  a = pool.take(0);
  pool.leave();
  CHECK(alive == 1);
  pool.give(std::move(a));   // nobody is left to lend it to
  CHECK(alive == 0 && !pool.take(0));
  std::vector<std::thread> th;
  for (int t = 0; t < 8; ++t)
    th.emplace_back([&, t] {
      for (int r = 0; r < 2000; ++r) {
        pool.enter();
        auto p = pool.take(t % 2);
        if (!p) p = std::make_unique<Thing>(t % 2);
        CHECK(p->device == t % 2 && p->held++ == 0);
        p->held--;
        pool.give(std::move(p));
        pool.leave();
      }
    });
  for (auto& x : th) x.join();
  CHECK(alive == 0);
}
""")
