"""CPU: the streaming loop's rules on ring rows (stream_plan.h, built with the host compiler).

For windows at the kernels' limits, every chunk start and every ring the rows that a kernel stages, written out here page by page as the
kernels stage them, are set against the rules: stream_ring_lo and stream_halo cover them all, and an update that
stream_apart lets run beside the attention writes none of their slots.
"""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "butterfly_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "stream_plan.h"
using namespace bfly;

// Lowest ring position staged for queries [q0, q0 + n): attn_mfma_kernel stages each query page and the one
// before it, page_attn_kernel the pages that hold a window key of the page's first query, win_attn_kernel
// the 192 positions up to the query page's end.
static long staged_lo(StreamKernel k, long q0, long n, long W) {
  long lo = q0;
  for (long page = q0 / 64; page <= (q0 + n - 1) / 64; ++page) {
    const long first = page * 64 > q0 ? page * 64 : q0;
    long x = page * 64 - 64;
    if (k == StreamKernel::kWindow) x = page * 64 - 128;
    if (k == StreamKernel::kPaged) x = first - W + 1 > 0 ? (first - W + 1) / 64 * 64 : 0;
    lo = x < lo ? x : lo;
  }
  return lo > 0 ? lo : 0;
}

int main() {
  const struct {
    StreamKernel k;
    std::vector<long> windows;
  } kernels[] = {
      {StreamKernel::kMfma, {1, 2, 33, 63, 64}},
      {StreamKernel::kWindow, {65, 66, 100, 127, 128}},
      {StreamKernel::kPaged, {1, 2, 64, 65, 129, 300}}};
  long checked = 0;
  for (const auto& kk : kernels)
    for (long W : kk.windows) {
      const long halo = stream_halo(kk.k, W);
      for (long q0 = 700; q0 < 764; ++q0)
        for (long cur : {1L, 64L, 100L}) {
          const long lo = staged_lo(kk.k, q0, cur, W);
          if (lo < stream_ring_lo(kk.k, q0, W) || lo < q0 - halo) {
            std::printf("kernel %d W %ld q0 %ld: stages %ld, rule %ld, halo %ld\n", (int)kk.k, W, q0, lo,
                        (long)stream_ring_lo(kk.k, q0, W), halo);
            return 1;
          }
          for (long next : {1L, 130L})
            for (long ring = cur + next; ring < cur + next + halo + 3; ++ring) {
              // slots written for [q0 + cur, + next) against the slots of [lo, q0 + cur), one by one
              std::vector<char> read(ring, 0);
              bool clash = false;
              for (long p = lo; p < q0 + cur; ++p) read[p % ring] = 1;
              for (long p = q0 + cur; p < q0 + cur + next; ++p) clash = clash || read[p % ring];
              if (clash && stream_apart(cur, next, halo, ring)) {
                std::printf("kernel %d W %ld q0 %ld cur %ld next %ld ring %ld share a slot\n", (int)kk.k, W, q0, cur, next, ring);
                return 1;
              }
              if (ring_disjoint(q0 + cur, q0 + cur + next, lo, q0 + cur, ring) == clash) {
                std::printf("ring_disjoint W %ld q0 %ld cur %ld next %ld ring %ld\n", W, q0, cur, next, ring);
                return 1;
              }
              ++checked;
            }
        }
    }
  std::printf("%ld\n", checked);
  return 0;
}
"""


def test_updates_beside_attention_take_other_slots(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no host compiler")
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = tmp_path / "plan"
    subprocess.run([gxx, "-std=c++17", "-O2", "-I", str(CSRC), str(tmp_path / "main.cpp"), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout
    assert int(done.stdout) > 100_000
