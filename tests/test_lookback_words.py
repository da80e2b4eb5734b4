"""CPU: a run of a direct encode that leaves a record out of the container says so, in whatever order its
workgroups start and end.  The words and what the kernel does to them (neuzip_amd/csrc/nz_lookback.h) are compiled
for the host and taken through every order of four workgroups, from scratch memory with and without the abort mark."""
import os
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include "nz_lookback.h"

enum { N = 4 };                 // workgroups; the last one has the last chunk
static long orders, marked, late_starts;

struct Run {
  NzLbWords w;
  uint32_t runs[N], abort[N];   // what each read when it started
  int at[N];                    // 0: not started, 1: running, 2: ended
  bool left_out;
};

static int walk(const Run& r, uint64_t nonce, unsigned gives_up) {
  bool any = false;
  for (int i = 0; i < N; ++i) {
    if (r.at[i] == 2) continue;
    any = true;
    Run q = r;
    const bool last = i == N - 1;
    if (r.at[i] == 0) {
      q.runs[i] = q.w.runs;
      q.abort[i] = q.w.abort;
      q.at[i] = 1;
      if (r.at[N - 1] == 2) ++late_starts;
    } else {
      q.at[i] = 2;
      if (q.abort[i] == NZ_LOOKBACK_ABORT) {
        nz_lb_unplaced(&q.w, nonce, q.runs[i], last);
        q.left_out = true;
      } else if (gives_up >> i & 1) {
        nz_lb_gave_up(&q.w, nonce, q.runs[i], last);
        q.left_out = true;
      } else {
        nz_lb_placed(&q.w, q.runs[i], last);
        if (gives_up >> (N + i) & 1) {  // a record that does not fit
          nz_lb_left_out(&q.w, nonce);
          q.left_out = true;
        }
      }
    }
    if (int rc = walk(q, nonce, gives_up)) return rc;
  }
  if (!any) {
    ++orders;
    marked += r.left_out;
    if (nz_lb_not_whole(&r.w, nonce) != r.left_out) return 1;
  }
  return 0;
}

int main() {
  for (uint32_t abort : {0u, NZ_LOOKBACK_ABORT})
    for (uint32_t runs : {0u, 7u, 0xFFFFFFFFu})
      for (unsigned gives_up = 0; gives_up < 1u << N; ++gives_up)
        for (unsigned tight : {0u, 1u << N, 1u << (2 * N - 1)}) {
          if (gives_up & 1) continue;  // the first chunk waits for nobody
          Run r;
          memset(&r, 0, sizeof r);
          r.w.runs = runs, r.w.abort = abort, r.w.left_out = 0x1234567800000000ull | (runs + 1u);
          if (int rc = walk(r, 0x9E3779B97F4A7C15ull, gives_up | tight)) {
            printf("abort %x runs %x gives_up %x\n", abort, runs, gives_up | tight);
            return rc;
          }
        }
  printf("%ld orders, %ld with a record left out, %ld starts behind the last chunk's end\n", orders, marked, late_starts);
  return !(orders > 100000 && marked > 1000 && orders > marked && late_starts > 1000);
}
"""


def test_a_record_left_out_is_marked_in_every_order(tmp_path):
    (tmp_path / "walk.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror=return-type", "-I", os.path.join(ROOT, "neuzip_amd", "csrc"),
                    "-o", str(tmp_path / "walk"), str(tmp_path / "walk.cpp")], check=True)
    res = subprocess.run([str(tmp_path / "walk")], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
