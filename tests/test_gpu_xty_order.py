"""Weight gradients in every class of tiles under loads that differ: the order that gives each XCD its share of every expert,
super tiles for even loads and for more experts than that order sorts; 256 x 128 tiles two workgroups per CU, whose contraction
ends anywhere.  Every output is written (they start as NaN) and every class is within one rounding of float64."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _loads(E, rows, kind):
    if kind == "even":
        return [rows] * E
    if kind == "last":                                     # everything in the last experts, the others empty or nearly
        loads = [0, 1, 0, 63, 65, 2] * (E // 6 + 1)
        loads = loads[:E]
        loads[-1] = 0
        loads[-1] = E * rows - sum(loads)
        return loads
    loads = [max(0, int(E * rows * 0.5 ** (i + 1)) // 2 * 2 - 1) for i in range(min(E, 10))] + [0] * max(0, E - 10)      # odd, halves
    loads = loads[::-1]
    loads[0] += E * rows - sum(loads)
    return loads


def _run(E, K, N, rows, kind, layout, gather, bias, dtype):
    g = torch.Generator(device=DEV).manual_seed(E + K + N)
    loads = _loads(E, rows, kind)
    L, k = sum(loads), 2
    assert L == E * rows and L % k == 0 and min(loads) >= 0
    off = torch.cumsum(torch.tensor(loads), 0).to(DEV)
    DY = torch.randn(L, N, generator=g, device=DEV).to(dtype)
    X = torch.randn(L // k if gather else L, K, generator=g, device=DEV).to(dtype)
    idx = torch.randperm(L, generator=g, device=DEV)
    shape = (E, K, N) if layout == "kn" else (E, N, K)
    DW = torch.full(shape, float("nan"), device=DEV, dtype=dtype)
    DW = DW if layout == "kn" else DW.permute(0, 2, 1)
    Db = torch.full((E, N), float("nan"), device=DEV, dtype=dtype) if bias else None
    if gather:
        assert ops._backend.xty_gathered(DY, X, idx, k, DW, Db, off, E)
        X = X[idx // k]
    else:
        ops._backend.xty(DY, X, DW, Db, off, E)
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    lo = 0
    for e, n in enumerate(loads):
        x, y = X[lo:lo + n].double(), DY[lo:lo + n].double()
        # one rounding to the storage type, float32 sums of n products in any order
        for got, want, mass in ((DW[e], x.t() @ y, x.abs().t() @ y.abs()),
                                (Db[e] if bias else None, y.sum(0), y.abs().sum(0))):
            if got is not None:
                bound = unit * want.abs() + n * 2.0 ** -24 * mass + 2.0 ** -24
                assert bool(((got.double() - want).abs() <= bound).all()), (e, n)
        lo += n


# 256 x 128 tiles: 240 of 256 x 256, less than a round of two workgroups per CU; columns and rows of the last tiles partly filled
@pytest.mark.parametrize("kind", ["even", "last", "halves"])
@pytest.mark.parametrize("layout,gather,bias", [("nk", False, True), ("nk", True, True), ("kn", True, False), ("kn", False, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_pairs(kind, layout, gather, bias, dtype):
    _run(8, 1288, 1032, 298, kind, layout, gather, bias, dtype)


# (252 of 256 x 256: 256 x 128 tiles up to 2046 rows, eight waves at 2048; 264 leave the chip idle in a second round and go in small
# tiles)
@pytest.mark.parametrize("E,K,N", [(4, 2056, 1544), (2, 2824, 2568)])
@pytest.mark.parametrize("rows", [96, 257, 700, 2046, 2047])
def test_pairs_remainders(rows, E, K, N):
    _run(E, K, N, rows + rows % 2, "halves", "nk", True, True, torch.bfloat16)


# more than a round of 256 x 128 tiles, beyond what goes in small ones
def test_pairs_of_more_rounds():
    _run(12, 2056, 1544, 1200, "halves", "kn", False, True, torch.bfloat16)


# small tiles (few rows; two rounds of the larger ones; a second one partly filled), eight waves (gathered, 2048 rows), one wave per SIMD
@pytest.mark.parametrize("E,K,N,rows,gather", [(30, 264, 136, 100, True), (8, 2056, 1544, 400, True), (2, 3080, 2568, 2048, False),
                                               (3, 3080, 5128, 2048, True), (4, 2056, 1544, 2048, False)])
@pytest.mark.parametrize("kind", ["even", "last", "halves"])
@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_other_classes(E, K, N, rows, gather, kind, layout):
    _run(E, K, N, rows, kind, layout, gather, False, torch.bfloat16)


# one group of 64 experts exactly, two, the most that are sorted, one more
@pytest.mark.parametrize("E", [1, 2, 64, 65, 130, 256, 257])
@pytest.mark.parametrize("kind", ["last", "halves"])
@pytest.mark.parametrize("K,rows", [(136, 100), (392, 258)])      # super tiles whatever the loads; by rows
def test_numbers_of_experts(E, K, rows, kind):
    _run(E, K, 264, rows, kind, "nk", True, True, torch.bfloat16)
