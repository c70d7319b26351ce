"""The order of a launch's tiles in column stripes (Raster::map in csrc/gemm_mfma.hpp), asked of the code itself in a host-only
build: every tile is somebody's, and no XCD has more of them than its share."""
import ctypes
import os
import shutil
import subprocess

import pytest

from scattermoe_amd import _build

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")

SOURCE = """
#include <hip/hip_runtime.h>
#undef __global__
#define __global__ static __device__ __attribute__((unused))
#undef __launch_bounds__
#define __launch_bounds__(...)
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...)
#include "%(csrc)s/gemm_mfma.hpp"
using namespace smoe;
// tiles of workgroup ids 0, 1, ... as row * 65536 + column, -1 for a workgroup without one; their number
extern "C" int64_t stripes(int64_t m_tiles, int n_tiles, int* tiles) {
  const Raster r = make_striped(m_tiles, n_tiles, GM_RING);
  for (int64_t p = 0; p < r.grid(); ++p) {
    int m, n, ml, nl;
    tiles[p] = r.map((int)p, m, n, ml, nl) ? m * 65536 + n : -1;
  }
  return r.grid();
}
extern "C" int stripes_group() { return GM_RING; }
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    src, lib = d / "order.hip", d / "order.so"
    src.write_text(SOURCE % {"csrc": _build.CSRC})
    subprocess.run([_build._hipcc(), "--cuda-host-only", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-shared",
                    "-Wno-unused-command-line-argument", "-o", str(lib), str(src)], check=True)
    lib = ctypes.CDLL(str(lib))
    lib.stripes.restype = ctypes.c_int64
    return lib


@pytest.mark.parametrize("n_tiles", [1, 2, 7, 8, 9, 11, 12, 15, 16, 17, 22, 28])
def test_stripes_share_the_tiles_out(order, n_tiles):
    for m_tiles in (1, 7, 8, 9, 35, 51, 64, 133):
        buf = (ctypes.c_int * (8 * (m_tiles + 16) * (n_tiles + 8)))()
        grid = order.stripes(ctypes.c_int64(m_tiles), n_tiles, buf)
        tiles = [(x % 8, t // 65536, t % 65536) for x, t in enumerate(buf[:grid]) if t >= 0]
        assert sorted(t[1:] for t in tiles) == [(m, n) for m in range(m_tiles) for n in range(n_tiles)]
        gm = min(order.stripes_group(), m_tiles)
        # The rows that there are, up to the bound that the grid covers: an XCD's columns of all whole groups of rows differ by one
        # from its share at the most, and so do those of the last group
        for rows in range(1, m_tiles + 1):
            whole, rest = divmod(rows, gm)
            per_xcd = [sum(x == xcd and m < rows for x, m, _ in tiles) for xcd in range(8)]
            assert max(per_xcd) <= -(-whole * n_tiles // 8) * gm + -(-n_tiles // 8) * rest, (m_tiles, rows, per_xcd)


@pytest.mark.parametrize("n_tiles", [1, 3, 4, 8, 12, 22])
def test_stripes_leave_no_gaps(order, n_tiles):
    """An XCD's workgroups all have a tile until its last one of the whole groups of rows."""
    for m_tiles in (8, 40, 136):
        buf = (ctypes.c_int * (8 * (m_tiles + 16) * (n_tiles + 8)))()
        grid = order.stripes(ctypes.c_int64(m_tiles), n_tiles, buf)
        assert m_tiles * n_tiles <= grid < m_tiles * n_tiles + 8 * order.stripes_group()
        for xcd in range(8):
            has = [t >= 0 for t in buf[xcd:grid:8]]
            assert all(has[:sum(has)]), (m_tiles, xcd)
