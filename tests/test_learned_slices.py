"""The slices of a training batch (csrc/learned_slices.h): a workspace made for a batch has room for the
partials of every smaller batch, which run in it without allocating again."""
import ctypes
import os
import subprocess

import pytest

from fosolvers_amd import build as B

PROBE = """
#include "learned_slices.h"
extern "C" {
long rows(long n) { return (long)fos::slice_rows(n); }
long count(long n) { return (long)fos::slice_count(n); }
long room(long n) { return (long)fos::slice_room(n); }
// the first n in (1, last) whose room is short of a batch of at most n rows, or 0
long short_at(long last) {
  size_t most = 0;
  for (long n = 1; n <= last; n++) {
    if (fos::slice_count(n) > most) most = fos::slice_count(n);
    if (fos::slice_room(n) < most) return n;
  }
  return 0;
}
// the first n whose slices do not cover it, or leave the last one empty, or 0
long uncovered_at(long last) {
  for (long n = 1; n <= last; n++) {
    const size_t r = fos::slice_rows(n), k = fos::slice_count(n);
    if (k * r < (size_t)n || (k - 1) * r >= (size_t)n || r % 32 || k > 256) return n;
  }
  return 0;
}
}
"""


@pytest.fixture(scope="module")
def slices(tmp_path_factory):
    d = tmp_path_factory.mktemp("slices")
    src, so = d / "probe.cpp", d / "probe.so"
    src.write_text(PROBE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", B.CSRC, str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(os.fspath(so))
    for f in (lib.rows, lib.count, lib.room, lib.short_at, lib.uncovered_at):
        f.restype, f.argtypes = ctypes.c_long, [ctypes.c_long]
    return lib


def test_slices_cover_every_batch(slices):
    assert slices.uncovered_at(8_000_000) == 0


def test_room_covers_every_smaller_batch(slices):
    """Above 131,072 rows the rows per slice grow in steps of 32 and a smaller batch can have more slices:
    140,000 rows are 244 slices and 130,000 are 254."""
    for big, small in ((140_000, 130_000), (200_000, 196_000), (131_073, 131_072), (131_073, 130_112)):
        assert slices.count(small) > slices.count(big)
        assert slices.room(big) >= slices.count(small), (big, small)
    assert slices.short_at(8_000_000) == 0


def test_room_is_bounded(slices):
    """What a batch asks for beyond its own slices: nothing up to 131,072 rows, never more than 256."""
    assert all(slices.room(n) == slices.count(n) for n in (1, 511, 512, 513, 65_536, 131_072))
    assert max(slices.room(n) for n in (131_073, 1_500_000, 6_000_000)) == 256
