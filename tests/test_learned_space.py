"""The learned preconditioner's row buffers (csrc/learned_space.h) with an allocator that fails on request:
a call after a failed one finds every buffer it uses in place, or fails again; set-up and apply hold what
they use and no more; training leaves their buffers where they are."""
import ctypes
import os
import subprocess

import pytest

from fosolvers_amd import build as B

PROBE = """
#include <cstdlib>
#include "learned_space.h"
static long calls, failAt, bytes;
template <class T>
struct Buf {  // DBuf's behaviour: alloc frees first, and a failure leaves the buffer empty
  T *p = nullptr;
  size_t n = 0;
  int alloc(size_t count) {
    bytes -= (long)(n * sizeof(T));
    p = nullptr;
    n = 0;
    if (++calls == failAt) return -1;
    p = reinterpret_cast<T *>(64 * calls);  // never read; another address each time
    n = count;
    bytes += (long)(n * sizeof(T));
    return 0;
  }
  bool holds(size_t count) const { return p && n >= count; }
};
struct Space : fos::LearnedSpace<Buf> {
  bool has_apply(size_t n) const {
    return H0.holds(128 * n) && H1.holds(128 * n) && O.holds(32 * n) && t.holds(12 * n) && kappa.holds(n) &&
           red.holds(768);
  }
  bool has_inputs(size_t n) const { return X.holds(32 * n) && red.holds(768); }
  bool has_train(size_t n) const {
    return has_inputs(n) && HM0.holds(256 * n) && HM1.holds(256 * n) && H2.holds(128 * n) && O.holds(32 * n) &&
           t.holds(12 * n) && kappa.holds(n) && pre0.holds(128 * n) && pre1.holds(128 * n) && pre2.holds(128 * n) && rh.holds(8 * n) &&
           e.holds(8 * n) && ds.holds(8 * n) && part.holds(fos::slice_count(n) * fos::NPART) && dO16.holds(32 * n) &&
           dP.holds(128 * n) && dX.holds(256 * n) && bnbr.holds(4 * n) && red.holds((n + 255) / 256);
  }
};
extern "C" {
// allocation number fail of an inputs, a training and a set-up call fails; then the three calls again.
// Returns a bit per call that said yes without its buffers, and -1 when none failed.
int after_failure(long rows, long cells, long fail) {
  Space s;
  calls = 0;
  failAt = fail;
  int bad = (s.inputs(cells) == 0) != s.has_inputs(cells) ? 1 : 0;
  bad |= (s.train(rows) == 0) != s.has_train(rows) ? 1 : 0;
  bad |= (s.apply(cells) == 0) != s.has_apply(cells) ? 1 : 0;
  if (calls < fail) return -1;
  failAt = 0;
  bad |= s.apply(cells) || !s.has_apply(cells) ? 2 : 0;
  bad |= s.train(rows) || !s.has_train(rows) ? 4 : 0;
  bad |= s.inputs(cells) || !s.has_inputs(cells) ? 8 : 0;
  return bad;
}
// a second call of the same or smaller sizes allocates nothing
long again(long rows, long cells) {
  Space s;
  failAt = 0;
  if (s.apply(cells) || s.inputs(cells) || s.train(rows)) return -1;
  calls = 0;
  for (long n = rows; n > 0; n = n * 7 / 8)
    if (s.train(n)) return -1;
  return s.apply(cells) || s.inputs(cells) ? -1 : calls;
}
// the bytes that set-up and apply hold
long apply_bytes(long cells) {
  Space s;
  failAt = bytes = 0;
  return s.apply(cells) ? -1 : bytes;
}
// whether training after a set-up moves a buffer that the set-up and the apply write
int training_moves(long rows, long cells) {
  Space s;
  failAt = 0;
  if (s.apply(cells)) return -1;
  const void *was[] = {s.O.p, s.t.p, s.kappa.p, s.red.p, s.H0.p, s.H1.p};
  if (s.inputs(cells) || s.train(rows)) return -1;
  const void *is[] = {s.O.p, s.t.p, s.kappa.p, s.red.p, s.H0.p, s.H1.p};
  for (int k = 0; k < 6; k++)
    if (was[k] != is[k]) return 1;
  return 0;
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
    lib.apply_bytes.restype, lib.apply_bytes.argtypes = L, [L]
    lib.training_moves.restype, lib.training_moves.argtypes = ctypes.c_int, [L, L]
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


@pytest.mark.parametrize("cells", [262_144, 1_500_000, 6_000_000])
def test_set_up_and_apply_hold_what_they_use(space, cells):
    """Two hidden layers of 128 BF16 values, 32 outputs, t and its weights, the output scale: 692 bytes a
    cell, beside the reductions."""
    assert cells * 692 <= space.apply_bytes(cells) <= cells * 692 + 8 * (cells // 256 + 1024)


@pytest.mark.parametrize("rows,cells", [(1, 6), (65_536, 1_500_000), (1_000_000, 1_500_000), (1_500_000, 1_500_000)])
def test_training_leaves_the_set_up_where_it_is(space, rows, cells):
    assert space.training_moves(rows, cells) == 0
