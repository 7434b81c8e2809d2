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
