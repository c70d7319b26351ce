"""Which tiles a launch goes in, asked of the launchers' own rules: a host-only build of the kernels' header (no GPU, no device
code).  The lines that a launch must not cross, each with the launch that was slower beyond it, and the classes that the GPU tests
mean to run."""
import ctypes
import os
import random
import shutil
import subprocess

import pytest

from scattermoe_amd import _build

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")

# Launches are noted (the launching function's name with its tile, the kernel, the workgroups) instead of being made.
SOURCE = """
#include <hip/hip_runtime.h>
#include <string>
static std::string launched;
static void note(const char* from, const char* kernel, unsigned grid) {
  launched += std::string(from) + " / " + kernel + " / " + std::to_string(grid) + "\\n";
}
#undef __global__
#define __global__ static __device__ __attribute__((unused))
#undef __launch_bounds__
#define __launch_bounds__(...)
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, ...) note(__PRETTY_FUNCTION__, #kernel, dim3(grid).x)
#include "%(csrc)s/gemm_mfma.hip"
#include "%(csrc)s/gemm_mfma_xty.hip"
#include "%(csrc)s/gemm_f32.hip"
namespace smoe {
int launch_status(const char*) { return 0; }
void set_error(const char*, ...) {}
int dispatch_s2s_f16(const S2SArgs&, bool, hipStream_t) { return 0; }
bool try_s2s_rowdot(const S2SArgs&, int, hipStream_t, int&) { return false; }
}
using namespace smoe;
static void* at(int64_t offset) { return (void*)(0x10000 + offset); }
static S2SArgs s2s_args(int64_t E, int64_t K, int64_t N, int64_t L, int n_contiguous, int64_t pad) {
  S2SArgs a{};
  a.X = at(0), a.W = at(0), a.Y = at(0);
  a.E = (int)E, a.K = (int)K, a.N = (int)N, a.L = (int)L, a.fan_out = 1, a.x_grouped = a.y_grouped = 1;
  a.sxk = a.syn = 1, a.sxm = K + pad, a.sym = N;
  if (n_contiguous) a.swn = 1, a.swk = N + pad, a.swe = K * (N + pad);
  else a.swk = 1, a.swn = K + pad, a.swe = N * (K + pad);
  return a;
}
extern "C" const char* s2s_launch(int64_t E, int64_t K, int64_t N, int64_t L, int n_contiguous, int64_t expanded) {
  launched.clear();
  S2SArgs a = s2s_args(E, K, N, L, n_contiguous, 0);
  if (expanded) a.swk = 0;
  dispatch_s2s<bf16_t>(a, n_contiguous, 0);
  return launched.c_str();
}
extern "C" const char* s2s_f32_launch(int64_t E, int64_t K, int64_t N, int64_t L, int n_contiguous, int64_t pad) {
  launched.clear();
  int rc;
  if (!try_s2s_f32(s2s_args(E, K, N, L, n_contiguous, pad), 0, rc)) launched = "any layout";
  return launched.c_str();
}
extern "C" int s2s_pairs(int64_t K, int64_t N, int glu, int64_t pitch, int64_t h_pitch, int64_t y_at, int saved) {
  S2SArgs a{};
  a.K = (int)K, a.N = (int)N, a.glu = glu;
  a.Y = saved ? at(y_at) : nullptr, a.H = at(0), a.aux = at(0);
  a.sym = a.saux = pitch, a.shm = h_pitch;
  return takes_pairs(a);
}
static XtYArgs xty_args(int64_t E, int64_t K, int64_t N, int64_t L, int gathered, int n_contiguous) {
  XtYArgs a{};
  a.DY = at(0), a.X = at(0), a.DW = at(0), a.off = (const int64_t*)at(0);
  a.E = (int)E, a.K = (int)K, a.N = (int)N, a.L = (int)L;
  a.sdyn = a.sxk = 1, a.sdym = N, a.sxm = K, a.sdwe = K * N;
  a.sdwk = n_contiguous ? N : 1, a.sdwn = n_contiguous ? 1 : K;
  if (gathered) a.idx = (const int64_t*)at(0), a.fan_out = 2;
  return a;
}
extern "C" int xty_tiles(int64_t E, int64_t K, int64_t N, int64_t L, int gathered, int bias, int n_contiguous, int64_t dy_pitch,
                         int64_t x_pitch) {
  XtYArgs a = xty_args(E, K, N, L, gathered, n_contiguous);
  a.Db = bias ? at(0) : nullptr, a.sdym = dy_pitch, a.sxm = x_pitch;
  return (int)xty_class(a);
}
extern "C" int xty_gathers(int64_t E, int64_t K, int64_t N, int64_t L, int n_contiguous) {
  int rc;
  return try_xty_mfma(xty_args(E, K, N, L, 1, n_contiguous), SMOE_BF16, 0, rc);
}
extern "C" const char* xty_f32_launch(int64_t E, int64_t K, int64_t N, int64_t L, int64_t pad) {
  launched.clear();
  XtYArgs a{};
  a.DY = at(0), a.X = at(0), a.DW = at(0);
  a.E = (int)E, a.K = (int)K, a.N = (int)N, a.L = (int)L;
  a.sdyn = a.sxk = a.sdwk = 1, a.sdym = N + pad, a.sxm = K + pad, a.sdwn = K, a.sdwe = N * K;
  int rc;
  if (!try_xty_f32(a, 0, rc)) launched = "any layout";
  return launched.c_str();
}
extern "C" int64_t xty_workgroups(int64_t E, int64_t np, int64_t nq, int64_t L, int wide) {
  XtYPlan p{};
  p.E = (int)E, p.np = (int)np, p.nq = (int)nq;
  int64_t grid;
  if (wide) xty_order<Tile<256, 256, 2, 4>>(p, L, grid);
  else xty_order<Tile<128, 128, 2, 2, 1, false, 4>>(p, L, grid);
  return grid;
}
"""
XTY_CLASSES = ("held", "small", "pairs", "one wave", "large")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, lib = d / "rules.hip", d / "rules.so"
    src.write_text(SOURCE % {"csrc": _build.CSRC})
    subprocess.run([_build._hipcc(), "--cuda-host-only", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-shared",
                    "-Wno-unused-command-line-argument", "-o", str(lib), str(src)], check=True)
    lib = ctypes.CDLL(str(lib))
    lib.xty_workgroups.restype = ctypes.c_int64
    lib.s2s_launch.restype = lib.s2s_f32_launch.restype = lib.xty_f32_launch.restype = ctypes.c_char_p
    return lib


def _pairs(rules, K, N, glu=0, pitch=None, y_at=0, saved=True):
    width = 2 * N if glu in (1, 2, 4) else N
    return bool(rules.s2s_pairs(*(ctypes.c_int64(v) for v in (K, N)), glu, ctypes.c_int64(pitch or width),
                                ctypes.c_int64(N // 2 if glu == 3 else N), ctypes.c_int64(y_at), int(saved)))


@pytest.mark.parametrize("glu", [1, 2])
def test_gated_products_of_ragged_rows_keep_wide_tiles(rules, glu):
    """Rows that are no whole number of 64-byte pieces share one at every edge of a tile (64 experts x 230 rows, 64 -> 6952: 325
    us in 256 x 256 tiles, 509 in 256 x 128)."""
    for K, N in ((64, 6952), (192, 2152), (1536, 592), (1728, 1000)):
        assert not _pairs(rules, K, N, glu), (K, N)
        assert _pairs(rules, K, N // 32 * 32, glu), (K, N)
    assert not _pairs(rules, 64, 2048, glu, y_at=32) and _pairs(rules, 64, 2048, glu, y_at=64)
    assert not _pairs(rules, 64, 2048, glu, pitch=4096 + 8)


def test_interleaved_gated_products(rules):
    assert _pairs(rules, 64, 2 * 2048, 3) and _pairs(rules, 64, 2064, 4)
    assert not _pairs(rules, 960, 2 * 2056, 3) and _pairs(rules, 1024, 2 * 2056, 3)
    assert not _pairs(rules, 128, 2056, 4) and _pairs(rules, 192, 2056, 4)


def test_forward_that_saves_nothing(rules):
    assert _pairs(rules, 64, 2048, 1, pitch=4096 + 8, saved=False)
    assert not _pairs(rules, 128, 2056, 1, saved=False) and _pairs(rules, 192, 2056, 1, saved=False)
    assert not _pairs(rules, 128, 2 * 2056, 3, saved=False) and _pairs(rules, 192, 2 * 2056, 3, saved=False)


def test_plain_products(rules):
    """Ragged rows cost a plain product of a short contraction as well (64 x 504 rows, 64 -> 2088: 64 -> 76 us)."""
    assert _pairs(rules, 64, 2048) and not _pairs(rules, 64, 2088) and not _pairs(rules, 128, 2088)
    assert _pairs(rules, 192, 2088) and _pairs(rules, 1728, 2088)
    assert not _pairs(rules, 1792, 2048)                    # the one-wave-per-SIMD form
    assert not _pairs(rules, 200, 2048)                     # whole 64-deep slices
    assert not _pairs(rules, 192, 2048, y_at=8)             # 16-byte pieces


def _xty(rules, E, K, N, rows, layout="nk", gathered=False, bias=False, dy_pitch=None, x_pitch=None):
    i64 = ctypes.c_int64
    return XTY_CLASSES[rules.xty_tiles(i64(E), i64(K), i64(N), i64(E * rows), int(gathered), int(bias), int(layout == "kn"),
                                       i64(N if dy_pitch is None else dy_pitch), i64(K if x_pitch is None else x_pitch))]


def test_weight_gradients_of_one_tile_column_keep_wide_tiles(rules):
    """Two tiles of 128 columns in place of one of 256 read the rows twice (200 x 389 rows, 2752 x 256: 177 -> 205 us)."""
    assert _xty(rules, 200, 256, 2752, 389) == "large" and _xty(rules, 200, 3072, 192, 765, "kn") == "large"
    assert _xty(rules, 200, 264, 2752, 389) == "pairs" and _xty(rules, 200, 3072, 264, 765, "kn") == "pairs"
    assert _xty(rules, 200, 128, 2752, 600) == "pairs"


def test_weight_gradients_of_one_tile_row_keep_wide_tiles(rules):
    """Gathered rows that are looked up for every 128 columns of a single tile row (64 x 857 rows, 176 x 2520: 98 -> 113 us); uneven loads
    of more experts than the order by rows looks through (300 x 663, 24 x 4168: 2490 -> 3070)."""
    assert _xty(rules, 64, 176, 2520, 857, "kn", gathered=True) == "large"
    assert _xty(rules, 64, 176, 2520, 857, "kn") == _xty(rules, 64, 264, 2520, 857, "kn", gathered=True) == "pairs"
    assert _xty(rules, 64, 2520, 176, 857, "nk", gathered=True) == "pairs"
    assert _xty(rules, 300, 4168, 24, 1200) == "large" and _xty(rules, 256, 4168, 24, 1200) == "pairs"


def test_weight_gradients_of_many_rows_keep_wide_tiles(rules):
    """200 x 3491 rows, 256 x 256: 121 us in 256 x 256 tiles, 137 in 256 x 128."""
    for gathered, bias in ((True, False), (False, True)):
        assert _xty(rules, 4, 2056, 1544, 2048, gathered=gathered, bias=bias) == "large"
        assert _xty(rules, 4, 2056, 1544, 2047, gathered=gathered, bias=bias) == "pairs"
    assert _xty(rules, 4, 2056, 1544, 2048) == "one wave"


def _f32(launch, *sizes):
    text = launch(*(ctypes.c_int64(v) for v in sizes)).decode()
    return "small" if "small_kernel" in text else "any layout" if text == "any layout" else "large"


def test_float32_products(rules):
    """Times of the launch in 32 x 32 tiles against the other kind that it would go in."""
    def tiles(E, K, N, rows, pad=0, n_contiguous=0):
        return _f32(rules.s2s_f32_launch, E, K, N, E * rows, n_contiguous, pad)
    assert tiles(8, 512, 512, 64) == tiles(8, 4096, 1024, 256) == "small"
    assert tiles(8, 1024, 4096, 256) == "large"
    # short contractions: 64 x 909 rows, 16 -> 168 24 -> 54 us; 16 x 2296, 48 -> 1248 109 -> 252
    assert tiles(64, 16, 168, 909, 1) == tiles(16, 48, 1248, 2296, 1) == tiles(128, 28, 420, 1962, 1) == "any layout"
    assert tiles(8, 32, 512, 1024) == "large" and tiles(8, 32, 512, 128) == tiles(8, 128, 512, 256) == "small"
    assert tiles(8, 256, 2048, 256, 1) == tiles(32, 768, 768, 4096, 1) == "small"
    assert tiles(8, 256, 4096, 4096, 1) == "any layout"
    assert tiles(8, 256, 2048, 256, 1, 1) == "small"


def test_float32_weight_gradients(rules):
    def tiles(E, K, N, rows, pad=0):
        return _f32(rules.xty_f32_launch, E, K, N, E * rows, pad)
    # 8 x 16 rows, 512 x 512 8 -> 11 us; 32 x 4, 1592 x 4368, rows of no whole 16 bytes, 452 -> 706
    assert tiles(8, 512, 512, 16) == "large" and tiles(8, 512, 512, 48) == "small"
    assert tiles(8, 256, 512, 1) == tiles(8, 128, 512, 16) == tiles(8, 256, 512, 1, 1) == "small"       # up to 1024 of them
    assert tiles(32, 1592, 4368, 4, 1) == tiles(8, 512, 512, 31, 1) == "any layout" and tiles(8, 512, 512, 32, 1) == "small"
    assert tiles(8, 1024, 1024, 4096) == "large" and tiles(8, 1024, 1024, 4096, 1) == "small"


def _workgroups(rules, E, np_, nq, rows, wide):
    return rules.xty_workgroups(*(ctypes.c_int64(v) for v in (E, np_, nq, E * rows)), int(wide))


def test_weight_gradients_that_keep_super_tiles(rules):
    """Up to 256 rows per expert, more experts than are looked through, one column of 256 wide tiles: no order by rows, which costs even
    loads a look at all experts per tile (8 x 200 rows, 256 x 20000: 6 %).  Such launches have the super tiles' grid only; the
    order by rows gives every expert a whole number of workgroups per XCD, eight for an expert of one tile."""
    small = 8 * 256 // 2                                    # super tiles of 8 x 4, of which one column exists
    assert _workgroups(rules, 256, 128, 128, 256, False) == small and _workgroups(rules, 256, 128, 128, 257, False) == 8 * 256
    assert _workgroups(rules, 256, 256, 256, 2000, True) == small
    for wide, tile in ((True, 256), (False, 128)):
        assert _workgroups(rules, 257, tile, 2 * tile, 300, wide) < 8 * 257
        # (each covers its own order)
        assert _workgroups(rules, 40, 9 * tile, 5 * tile, 256, wide) >= 40 * 45
        assert _workgroups(rules, 40, 9 * tile, 5 * tile, 257, wide) >= 40 * 48


def test_held_operand(rules):
    """One operand in registers: not for narrow panels (300 x 180 rows, 64 x 6080 231 -> 595 us under loads as 1 / rank^0.84), not with
    few experts, one of which has most of the rows when loads differ (8 x 209 rows, 256 x 25344: 53 -> 86)."""
    for layout in ("nk", "kn"):
        shape = lambda panel, other: (panel, other) if layout == "kn" else (other, panel)
        assert _xty(rules, 32, *shape(384, 2880), 188, layout) == "held" and _xty(rules, 32, *shape(320, 2880), 188, layout) == "small"
        assert _xty(rules, 16, *shape(2048, 1536), 96, layout) == "held" and _xty(rules, 16, *shape(2048, 1536), 95, layout) == "small"
        assert _xty(rules, 16, *shape(2048, 1536), 224, layout) == "held" and _xty(rules, 16, *shape(2048, 1536), 225, layout) == "small"
        assert _xty(rules, 15, *shape(4096, 2048), 188, layout) == "small"
        assert _xty(rules, 128, *shape(768, 64), 188, layout) == "held"


def test_wide_gradients_look_rows_up_only_where_they_are_streamed(rules):
    """Beyond 6144 columns the caller copies the gathered rows, unless they are streamed past the held operand."""
    def gathers(N, rows, layout):
        return bool(rules.xty_gathers(*(ctypes.c_int64(v) for v in (32, 2048, N, 32 * rows)), int(layout == "kn")))
    assert gathers(6144, 188, "nk") and gathers(6144, 188, "kn") and gathers(6144, 300, "kn")
    assert gathers(14336, 188, "nk") and not gathers(14336, 188, "kn") and not gathers(14336, 300, "nk")


def test_python_side_of_the_held_operand_agrees(rules):
    """The caller asks the same question before it decides on a copy (gradients with N contiguous, more than 512 tiles)."""
    from types import SimpleNamespace
    from scattermoe_amd.kernels import ops
    rng, held = random.Random(1), 0
    for _ in range(4000):
        E, rows = rng.choice((8, 15, 16, 17, 64)), rng.choice((95, 96, 150, 224, 225))
        K, N = rng.choice((376, 384, 1024, 2880)), rng.choice((2048, 2080, 2880, 6144))
        L = E * rows + rng.choice((0, rng.randrange(E)))
        L += L % 2
        x_pitch = K + rng.choice((0, 0, 8, 2 ** 30 // (L // 2) // 8 * 8))
        if E * -(-K // 256) * -(-N // 256) <= 512:
            continue
        DW = SimpleNamespace(shape=(E, K, N), stride=lambda i: (K * N, N, 1)[i])
        X = SimpleNamespace(size=lambda i: (L // 2, K)[i], stride=lambda i: (x_pitch, 1)[i])
        want = XTY_CLASSES[rules.xty_tiles(*(ctypes.c_int64(v) for v in (E, K, N, L)), 1, 0, 1, ctypes.c_int64(N),
                                           ctypes.c_int64(x_pitch))] == "held"
        assert ops._xty_holds_rows(DW, X, L) == want, (E, K, N, L, x_pitch)
        held += want
    assert 200 < held < 3000


@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_classes_that_the_gpu_tests_mean_to_run(rules, layout):
    """test_gpu_xty_order and test_gpu_expanded_operands: the loads differ there, the averages are these."""
    ask = lambda *sizes, **kw: _xty(rules, *sizes, layout, **kw)
    for gathered, bias in ((False, True), (True, True)):
        assert ask(8, 1288, 1032, 298, gathered=gathered, bias=bias) == "pairs"
    for rows in (258, 700, 2046):
        assert ask(4, 2056, 1544, rows, gathered=True, bias=True) == "pairs" and ask(2, 2824, 2568, rows, gathered=True, bias=True) == "small"
    assert ask(12, 2056, 1544, 1200, bias=True) == "pairs"
    assert ask(30, 264, 136, 100, gathered=True) == ask(8, 2056, 1544, 400, gathered=True) == ask(2, 3080, 2568, 2048) == "small"
    assert ask(3, 3080, 5128, 2048, gathered=True) == "large" and ask(4, 2056, 1544, 2048) == "one wave"
    for width in (64, 128, 192, 320):                      # test_gpu_xty_held
        K, N = (width, 512) if layout == "nk" else (512, width)
        assert ask(140, K, N, 148, gathered=True, bias=True) == "held"
    assert ask(20, 832, 1024, 148) == ask(20, 832, 1024, 148, dy_pitch=0) == ask(20, 832, 1024, 148, x_pitch=0) == "held"
    # rows on top of each other: neither descriptors that end with an operand's last row
    for rows, other in ((300, "pairs"), (2048, "one wave")):
        assert ask(4, 2056, 1544, rows) == other and ask(4, 2056, 1544, rows, dy_pitch=0) == ask(4, 2056, 1544, rows, x_pitch=0) == "large"


def test_overlapping_weights_leave_the_one_wave_form(rules):
    def tile(K, expanded):
        return rules.s2s_launch(*(ctypes.c_int64(v) for v in (2, K, 14336, 1200)), 1, ctypes.c_int64(expanded)).decode()
    assert "<256, 256, 2, 2, 2, true>" in tile(2048, 0) and "<256, 256, 2, 4>" in tile(2048, 1)
    assert "<256, 128, 2, 2, 2, false, 2, true>" in tile(1024, 0) and "<256, 128, 2, 2, 2, false, 2, true>" in tile(1024, 1)
