"""Which tiles products of few rows per expert, products in contraction parts and weight gradients of four rounds go in, asked of the
launchers' own rules as in test_dispatch_lines: each line from both sides, and the classes that the GPU tests mean to run."""
import ctypes
import subprocess

import pytest

from scattermoe_amd import _build
import test_dispatch_lines as lines
import test_gpu_narrow_tiles
import test_gpu_product_parts
import test_gpu_weights_once
import test_gpu_weights_once_wide as weights_once_wide
import test_gpu_xty_rounds

pytestmark = lines.pytestmark

SOURCE = lines.SOURCE + """
static S2SArgs fused_args(int64_t E, int64_t K, int64_t N, int64_t L, int n_contiguous, int glu) {
  const int64_t columns = glu == 1 ? 2 * N : N;
  S2SArgs a = s2s_args(E, K, columns, L, n_contiguous, 0);
  a.N = (int)N, a.glu = glu, a.H = at(0), a.aux = at(0);
  a.sym = a.saux = glu == 2 || glu == 4 ? 2 * N : columns, a.shm = glu == 3 ? N / 2 : N;
  return a;
}
extern "C" const char* product(int64_t E, int64_t K, int64_t N, int64_t L, int n_contiguous, int glu, int64_t workspace) {
  launched.clear();
  S2SArgs a = fused_args(E, K, N, L, n_contiguous, glu);
  if (workspace > 0) a.partial = (float*)at(0), a.partial_floats = workspace;
  dispatch_s2s<bf16_t>(a, n_contiguous, 0);
  return launched.c_str();
}
extern "C" int64_t workspace(int64_t E, int64_t K, int64_t N, int64_t L) { return s2s_workspace_floats(L, K, N, (int)E, SMOE_BF16); }
extern "C" int weights_once(int64_t E, int64_t K, int64_t N, int64_t L, int glu) {
  return reads_weights_once(fused_args(E, K, N, L, 0, glu));
}
"""
NARROW, WIDE, PAIRED = "<256, 192, 2, 2, 2, true>", "<256, 256, 2, 2, 2, true>", "<256, 128, 2, 2, 2, false, 2, true>"
LAYOUTS = {"k_contig": 0, "n_contig": 1}


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("products")
    src, lib = d / "products.hip", d / "products.so"
    src.write_text(SOURCE % {"csrc": _build.CSRC})
    subprocess.run([_build._hipcc(), "--cuda-host-only", "-x", "hip", "-std=c++17", "-O1", "-fPIC", "-shared",
                    "-Wno-unused-command-line-argument", "-o", str(lib), str(src)], check=True)
    lib = ctypes.CDLL(str(lib))
    lib.product.restype, lib.workspace.restype = ctypes.c_char_p, ctypes.c_int64
    return lib


def _i64(*sizes):
    return [ctypes.c_int64(v) for v in sizes]


def _launches(rules, E, K, N, L, layout="k_contig", glu=0, workspace=True):
    """The launches of a product, one line each; with the workspace that the caller is asked for."""
    need = rules.workspace(*_i64(E, K, N, L)) if workspace and glu == 0 else 0
    return rules.product(*_i64(E, K, N, L), LAYOUTS[layout], glu, ctypes.c_int64(need)).decode().splitlines()


def _parts(rules, E, K, N, L, **kw):
    """Contraction parts of a product (1: none)."""
    launches = _launches(rules, E, K, N, L, **kw)
    if len(launches) != 2 or "parts_sum_kernel" not in launches[1]:
        return 1
    assert WIDE in launches[0]
    parts, rest = divmod(rules.workspace(*_i64(E, K, N, L)), L * N)
    assert rest == 0
    return parts


def _only(rules, tile, *sizes, **kw):
    launches = _launches(rules, *sizes, **kw)
    return len(launches) == 1 and tile in launches[0]


@pytest.mark.parametrize("layout", LAYOUTS)
def test_tiles_of_192_columns(rules, layout):
    ask = lambda *sizes, glu=0: next((t for t in (NARROW, WIDE, PAIRED) if _only(rules, t, *sizes, layout=layout, glu=glu)), None)
    # 32 tile rows: 1.5 rounds of 256 columns, 1.9 of 192
    assert ask(32, 2880, 2880, 32 * 188) == ask(32, 2880, 2880, 32 * 188, glu=2) == ask(32, 2880, 2880, 32 * 188, glu=4) == NARROW
    assert ask(32, 2880, 2880, 32 * 188, glu=1) == ask(32, 2880, 2880, 32 * 188, glu=3) == WIDE      # forward units: 256
    assert ask(32, 2880, 3072, 32 * 188) == NARROW and ask(32, 2880, 3080, 32 * 188) == WIDE        # 512 tiles of 192; 544, a third round
    assert ask(64, 2048, 2064, 64 * 130) == NARROW and ask(64, 2048, 2048, 64 * 130) == WIDE        # three rounds; two, which become three
    assert ask(32, 2880, 2880, 32 * 224 - 1) == NARROW and ask(32, 2880, 2880, 32 * 224) == WIDE
    assert ask(32, 1792, 2880, 32 * 188) == NARROW and ask(32, 1728, 2880, 32 * 188) == PAIRED


def test_products_in_contraction_parts(rules):
    ask = lambda *sizes, **kw: _parts(rules, *sizes, **kw)
    assert ask(8, 14336, 4096, 8 * 194) == 2 and ask(1, 10240, 1472, 609) == 8
    assert ask(8, 14336, 4104, 8 * 194) == 1                 # 136 tiles: two parts would be a second round
    assert ask(8, 14336, 4096, 8 * 250) == 1                 # a third of the experts have a second tile row
    assert ask(8, 14336, 2048, 8 * 112) > 1 and ask(8, 14336, 2048, 8 * 112 - 1) == 1
    assert ask(8, 2048, 2048, 8 * 200) == 1                  # 32 slices: the sums cost more than the parts save
    assert ask(4, 14336, 4096, 1200) > 1 and ask(4, 14336 + 32, 4096, 1200) == 1        # whole slices
    assert ask(4, 14336, 4092, 1200) == 1                    # 16-byte pieces
    for glu in (1, 2, 3, 4):
        assert ask(8, 14336, 4096, 8 * 194, glu=glu) == 1
    assert ask(8, 14336, 4096, 8 * 194, workspace=False) == 1


def test_weights_that_bypass_the_caches(rules):
    ask = lambda *sizes, glu=0: bool(rules.weights_once(*_i64(*sizes), glu))
    assert ask(8, 4096, 5120, 8 * 194) and not ask(8, 4096, 5112, 8 * 194)              # 320 MB of weights
    assert ask(8, 4096, 2560, 8 * 194, glu=1) and not ask(8, 4096, 2560, 8 * 194, glu=3)      # N: one half's columns
    assert ask(8, 4096, 5120, 8 * 639) and not ask(8, 4096, 5120, 8 * 640)


def test_weight_gradients_with_one_wave_per_simd(rules):
    ask = lambda *sizes, **kw: lines._xty(rules, *sizes, **kw)
    # 8 experts x 11 x 12 tiles are four rounds and more, 8 x 11 x 11 are not
    assert ask(8, 2824, 2696, 1280) == ask(8, 2824, 2824, 1280) == "one wave"
    assert ask(8, 2824, 2824, 1279) == ask(8, 2696, 2696, 1280) == ask(8, 2696, 2696, 2047) == "pairs"
    assert ask(8, 2696, 2696, 2048) == "one wave" and ask(8, 2824, 2824, 1280, gathered=True) == "pairs"


@pytest.mark.parametrize("layout", LAYOUTS)
def test_classes_that_the_gpu_tests_mean_to_run(rules, layout):
    loads = test_gpu_narrow_tiles.LOADS * 2
    for N in (2880, 2696, 2872):
        for glu in (0, 2, 4):
            assert _only(rules, NARROW, len(loads), 1792, N, sum(loads) + 5, layout=layout, glu=glu), (N, glu)

    marks = test_gpu_product_parts.test_whole_products_in_contraction_parts.pytestmark
    cases = next(m.args[1] for m in marks if m.name == "parametrize" and m.args[0].startswith("loads"))
    for loads, dropped, K, N, parts in cases:
        got = _parts(rules, len(loads), K, N, sum(loads) + dropped, layout=layout)
        assert got > 1 and parts in (None, got), (loads, got)

    loads = test_gpu_weights_once.LOADS * 4                  # tiles of 192 columns, paired ones
    for (K, N), tile in (((2048, 1416), NARROW), ((1024, 2752), PAIRED)):
        assert _only(rules, tile, len(loads), K, N, sum(loads) + 5, layout=layout)
        assert rules.weights_once(*_i64(len(loads), K, N, sum(loads) + 5), 0)
    loads = weights_once_wide.LOADS * 4                      # tiles of 256 columns, one wave per SIMD
    K = weights_once_wide.K
    for N, glu in ((weights_once_wide.N, 0), (weights_once_wide.N, 2), (weights_once_wide.N, 3), (weights_once_wide.N, 4),
                   (weights_once_wide.N // 2, 1)):
        assert _only(rules, WIDE, len(loads), K, N, sum(loads) + 5, layout=layout, glu=glu), (N, glu)
        assert rules.weights_once(*_i64(len(loads), K, N, sum(loads) + 5), glu), (N, glu)
    loads, K, N = weights_once_wide.PARTS
    assert _parts(rules, len(loads), K, N, sum(loads) + 5, layout=layout) > 1 and rules.weights_once(*_i64(len(loads), K, N, sum(loads) + 5), 0)

    loads = [1280, 0, 1, 65, 2047, 1344, 2600, 2905]         # test_gpu_xty_rounds
    assert lines._xty(rules, 8, 2696, 2824, (sum(loads) + 5) // 8, {"k_contig": "nk", "n_contig": "kn"}[layout]) == "one wave"
    assert test_gpu_xty_rounds.DEV
