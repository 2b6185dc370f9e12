"""ringattn_jobs.h: quotients by reciprocal, and the jobs of a launch dealt to the workgroups of its grid -- every one of them to exactly
one, a head's to one XCD where heads deal out evenly, else in equal shares.  Compiled with the host compiler: it is the same
code as in the kernels."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdio.h>
#include <vector>
#include "ringattn_jobs.h"
using namespace ringattn;
int fails = 0;
#define CHECK(x, ...) do { if (!(x) && ++fails < 20) { printf("%s: ", #x); printf(__VA_ARGS__); printf("\n"); } } while (0)

void quotients(unsigned d) {
  const Divisor by = divisor(d);
  auto one = [&](int64_t n) { if (n >= 0 && n <= INT32_MAX) CHECK(quotient((int)n, by) == (int)(n / d), "%lld / %u", (long long)n, d); };
  for (int64_t n = 0; n < 300; ++n) one(n);
  for (int64_t k = 1; k < 40; ++k)   // around multiples near both ends of the range
    for (int64_t e = -1; e <= 1; ++e) { one(k * d + e); one(((int64_t)INT32_MAX / d - k + 1) * d + e); one(INT32_MAX - k); }
}

void jobs(int heads, int per_head, bool masked) {
  JobMap m;
  const int64_t blocks = job_map(m, heads, per_head, masked);
  CHECK(blocks % 8 == 0 && blocks < (int64_t)heads * per_head + 8 + 8 * heads, "%d heads x %d: %lld", heads, per_head, (long long)blocks);
  std::vector<int> seen((size_t)heads * per_head, 0), of_xcd(8, 0);
  for (int64_t b = 0; b < blocks; ++b) {
    int head = -1, job = -1;
    if (!job_of(m, masked, (int)(b & 7), (int)(b >> 3), head, job)) continue;
    CHECK(head >= 0 && head < heads && job >= 0 && job < per_head, "%d heads x %d, %d: head %d job %d", heads, per_head, masked, head, job);
    if (head < 0 || head >= heads || job < 0 || job >= per_head) return;
    if (head < (heads & ~7)) CHECK(head % 8 == (int)(b & 7), "head %d of %d on XCD %d", head, heads, (int)(b & 7));
    ++seen[(size_t)head * per_head + job];
    ++of_xcd[b & 7];
  }
  for (size_t i = 0; i < seen.size(); ++i) CHECK(seen[i] == 1, "%d heads x %d, %d: job %zu %d times", heads, per_head, masked, i, seen[i]);
  int lo = of_xcd[0], hi = of_xcd[0];
  for (int n : of_xcd) { lo = n < lo ? n : lo; hi = n > hi ? n : hi; }
  CHECK(hi - lo <= 7 && hi == blocks / 8, "%d heads x %d: %d to %d jobs an XCD", heads, per_head, lo, hi);
}

int main() {
  for (unsigned d = 1; d < 5000; ++d) quotients(d);
  for (unsigned l = 1; l < 31; ++l) for (int e = -2; e <= 2; ++e) if ((1u << l) + e >= 1) quotients((1u << l) + e);
  quotients(INT32_MAX);
  for (int masked = 0; masked < 2; ++masked)
    for (int heads = 1; heads <= 40; ++heads)
      for (int per_head : {1, 2, 3, 5, 7, 8, 15, 16, 31, 63, 64, 65, 128, 257, 1000}) jobs(heads, per_head, masked);
  for (int masked = 0; masked < 2; ++masked) { jobs(1, 400001, masked); jobs(7, 100003, masked); jobs(13, 30011, masked); jobs(1027, 3, masked); }
  printf("%d failures\n", fails);
  return fails != 0;
}
"""


def test_every_job_has_one_workgroup(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "jobs.cpp", tmp_path / "jobs"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-O1", "-std=c++17", "-I", os.path.join(ROOT, "ringattention_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
