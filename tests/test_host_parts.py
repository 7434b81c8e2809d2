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
    order of their ends; the events at hand stay below two for each of 256 spans and the open ones, and none is
    left. An event that cannot be made or recorded loses no other."""
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
    spans.resolve(SIZE_MAX, sink);
    CHECK(seen == 4 * 5700 + 1);
    CHECK(most <= 2 * (S::kMax + 3));
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
    spans.resolve(SIZE_MAX, [&](const S::Span&, float) { ++seen; });
    CHECK(ok == (f == 3 || f == 5 ? 3 : 2) && seen == 2);
  }
  CHECK(live.empty());
  return 0;
}
""")
