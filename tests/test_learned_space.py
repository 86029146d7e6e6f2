"""The learned preconditioner's row buffers (csrc/learned_space.h) with an allocator that fails on request:
a call after a failed one finds every buffer it uses in place, or fails again."""
import ctypes
import os
import subprocess

import pytest

from fosolvers_amd import build as B

PROBE = """
#include <cstdlib>
#include "learned_space.h"
static long calls, failAt;
template <class T>
struct Buf {  // DBuf's behaviour: alloc frees first, and a failure leaves the buffer empty
  T *p = nullptr;
  size_t n = 0;
  int alloc(size_t count) {
    p = nullptr;
    n = 0;
    if (++calls == failAt) return -1;
    p = reinterpret_cast<T *>(64);  // never read
    n = count;
    return 0;
  }
  bool holds(size_t count) const { return p && n >= count; }
};
struct Space : fos::LearnedSpace<Buf> {
  bool has_forward(size_t n) const {
    return X.holds(32 * n) && H0.holds(256 * n) && H1.holds(256 * n) && H2.holds(128 * n) && O.holds(32 * n) &&
           t.holds(12 * n) && kappa.holds(n) && red.holds(768);
  }
  bool has_train(size_t n) const {
    return has_forward(n) && pre0.holds(128 * n) && pre1.holds(128 * n) && pre2.holds(128 * n) && rh.holds(8 * n) &&
           e.holds(8 * n) && ds.holds(8 * n) && part.holds(fos::slice_count(n) * fos::NPART) && dO16.holds(32 * n) &&
           dP.holds(128 * n) && dX.holds(256 * n) && bnbr.holds(4 * n) && red.holds((n + 255) / 256);
  }
};
extern "C" {
// allocation number fail of a training call fails (0: none); then a training call, a forward call and the
// training call again.  Returns a bit per call that said yes without its buffers, and -1 when none failed.
int after_failure(long rows, long cells, long fail) {
  Space s;
  calls = 0;
  failAt = fail;
  const int first = s.train(rows);
  if (calls < fail) return -1;
  int bad = (first == 0) != s.has_train(rows) ? 1 : 0;
  failAt = 0;
  bad |= s.forward(cells) || !s.has_forward(cells) ? 2 : 0;
  bad |= s.train(rows) || !s.has_train(rows) ? 4 : 0;
  return bad;
}
// a second call of the same or smaller sizes allocates nothing
long again(long rows, long cells) {
  Space s;
  failAt = 0;
  if (s.forward(cells) || s.train(rows)) return -1;
  calls = 0;
  for (long n = rows; n > 0; n = n * 7 / 8)
    if (s.train(n)) return -1;
  return s.forward(cells) ? -1 : calls;
}
}
"""


@pytest.fixture(scope="module")
def space(tmp_path_factory):
    d = tmp_path_factory.mktemp("space")
    src, so = d / "probe.cpp", d / "probe.so"
    src.write_text(PROBE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", B.CSRC, str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(os.fspath(so))
    L = ctypes.c_long
    lib.after_failure.restype, lib.after_failure.argtypes = ctypes.c_int, [L, L, L]
    lib.again.restype, lib.again.argtypes = L, [L, L]
    return lib


@pytest.mark.parametrize("rows,cells", [(1, 1), (65_536, 65_536), (1_000, 200_000), (300_000, 300_000)])
def test_calls_after_a_failed_allocation(space, rows, cells):
    k = 1
    while (bad := space.after_failure(rows, cells, k)) >= 0:
        assert bad == 0, (k, bad)
        k += 1
    assert k > 10  # every allocation of the call has failed once


@pytest.mark.parametrize("rows,cells", [(1, 6), (65_536, 1_500_000), (140_001, 141_120)])
def test_buffers_are_kept(space, rows, cells):
    assert space.again(rows, cells) == 0
