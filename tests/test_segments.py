"""The dX kernels' walk over the segment table (csrc/gl_segments.h), compiled for the host: every edge of
a wave's unit range once, in order, wherever its rows lie in a table of up to 2^31 segments."""
import ctypes
import mmap
import shutil
import subprocess

import numpy as np
import pytest

from conftest import ROOT

HARNESS = """
#include <stdint.h>
#define __host__
#define __device__
#define __forceinline__ inline
namespace gl {
inline int opaque(int v) { return v; }
inline unsigned wave_uniform(unsigned v) { return v; }
}
#include "gl_segments.h"

// chunks of the walk as (unit, first edge, edges) rows; returns their number (at most cap)
extern "C" int walk(const uint32_t* seg_ptr, const int32_t* seg_unit, const uint32_t* seg_begin, int F, int u_lo,
                    int u_hi, int ahead, unsigned* out, int cap) {
  using namespace gl;
  const DxSegs s = dx_segs(seg_ptr, seg_unit, seg_begin, F, u_lo, u_hi);
  int n = 0;
  if (s.n <= 0) return 0;
  DxChunk c = dx_first(s);
  unsigned pe = 0, pu = 0;
  if (ahead) dx_seg_ahead(s, 0, pe, pu);
  while (c.si < s.n && n < cap) {
    const unsigned left = c.end - c.e;
    out[3 * n] = (unsigned)c.u, out[3 * n + 1] = c.e, out[3 * n + 2] = left < 64 ? left : 64;
    ++n;
    if (ahead) dx_next_ahead(s, c, pe, pu); else dx_next(s, c);
  }
  return n;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("segments")
    (d / "walk.cpp").write_text(HARNESS)
    subprocess.run([gxx, "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{ROOT}/granulelayer_amd/csrc", "-o",
                    str(d / "walk.so"), str(d / "walk.cpp")], check=True)
    return ctypes.CDLL(str(d / "walk.so")).walk


def table(rows):
    """uint32 array of `rows` entries in address space that takes memory only where it is written"""
    m = mmap.mmap(-1, rows * 4, flags=mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | 0x4000)  # MAP_NORESERVE
    return np.frombuffer(m, np.uint32)


# first row of the feature range: the table's start, either side of the row whose byte offset leaves 31
# and 32 bits, and the last rows of the largest table
@pytest.mark.parametrize("first", [0, 2**29 - 100, 2**30 - 100, 2**30 + 5, 2**31 - 301])
@pytest.mark.parametrize("ahead", [0, 1])
def test_walk_reaches_every_segment_of_a_large_table(walk, first, ahead):
    n, F = 300, 1
    rng = np.random.default_rng(first % 1000 + ahead)
    size = rng.choice([1, 2, 63, 64, 65, 130], n)
    unit, begin = table(2**31), table(2**31 + 1)
    units = np.sort(rng.choice(1000, n, replace=False))
    begins = 7 + np.concatenate([[0], np.cumsum(size)])
    unit[first:first + n] = units
    begin[first:first + n + 1] = begins
    seg_ptr = np.array([0, first, first + n], np.uint32)
    out = np.zeros((4 * n, 3), np.uint32)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    for u_lo, u_hi in ((0, 1000), (units[40], units[41]), (units[100] + 1, units[260]), (1000, 1100)):
        got = walk(ptr(seg_ptr), ptr(unit), ptr(begin), F, int(u_lo), int(u_hi), ahead, ptr(out), len(out))
        want = [(units[i], e, min(64, begins[i + 1] - e)) for i in range(n) if u_lo <= units[i] < u_hi
                for e in range(begins[i], begins[i + 1], 64)]
        assert out[:got].tolist() == [list(map(int, w)) for w in want]
