"""Weight gradients in small tiles (128 x 128, one operand stage): expert loads on both sides
of every slice boundary, output sizes that are no whole number of tiles, both output layouts, with and without
gathered rows and bias gradient, an output whose rows are not 16-byte aligned."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOADS = [1, 63, 64, 65, 0, 127, 128, 129, 191, 192, 193, 256, 300, 320, 31, 0]


def _check(got, want, mass, n, dtype):
    """One rounding to the storage type, float32 sums of n products of total magnitude `mass` in any order."""
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    bound = unit * want.abs() + n * 2.0 ** -24 * mass + 2.0 ** -24
    assert bool(((got.double() - want).abs() <= bound).all())


# 16 experts of 139 rows on average: few rows (512 output tiles of 256 x 256 and more); 64-wide sizes: few tiles
@pytest.mark.parametrize("K,N", [(2056, 1048), (1536, 1544), (200, 136), (64, 520)])
@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_against_float64(K, N, layout, dtype):
    g = torch.Generator(device=DEV).manual_seed(K + N)
    E, L, k = len(LOADS), sum(LOADS), 2
    loads = LOADS if L % k == 0 else LOADS[:-2] + [LOADS[-2] + 1, 0]
    L = sum(loads)
    experts = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(loads, device=DEV))
    experts = experts[torch.randperm(L, generator=g, device=DEV)].view(L // k, k)
    eid, idx, off = ops.route(experts, E)
    X = torch.randn(L // k, K, generator=g, device=DEV).to(dtype)
    DY = torch.randn(L, N, generator=g, device=DEV).to(dtype)
    like = torch.empty(E, K, N, dtype=dtype, device=DEV) if layout == "kn" else None
    Xg = ops.group(X, idx, fan_out=k)
    DW, Db = ops.group_bwd_W(DY, Xg, off, E, has_bias=True, like=like)
    DWg, Dbg = ops.group_bwd_W(DY, X, off, E, has_bias=True, like=like, gather=(idx, k))
    assert torch.equal(DW, DWg) and torch.equal(Db, Dbg)
    DWg, Dbg = torch.empty_like(DW), torch.empty_like(Db)
    assert ops._backend.xty_gathered(DY, X, idx, k, DWg, Dbg, off, E)          # rows looked up inside the launch
    assert torch.equal(DW, DWg) and torch.equal(Db, Dbg)
    ends = [0] + off.tolist()
    for e in range(E):
        x, y = Xg[ends[e]:ends[e + 1]].double(), DY[ends[e]:ends[e + 1]].double()
        n = x.size(0)
        _check(DW[e], x.t() @ y, x.abs().t() @ y.abs(), n, dtype)
        _check(Db[e], y.sum(0), y.abs().sum(0), n, dtype)


# both sides of the lines between small and 256 x 256 tiles where the chip would idle: at most 128 output tiles of 256 x 256
# (operands of 17 MB; of 270 MB with six tiles per expert, with four, with one), up to 160, a second round (400 tiles at the
# last row count of small tiles and the first of large ones); always rows enough for the one-wave-per-SIMD form
@pytest.mark.parametrize("E,rows,K,N", [(4, 2100, 520, 1040), (16, 8200, 520, 512), (32, 8200, 512, 512), (80, 2064, 256, 256),
                                        (40, 2100, 512, 512), (2, 1536, 2560, 5120), (2, 1537, 2560, 5120),
                                        (2, 2064, 2560, 5120)])
def test_many_rows(E, rows, K, N):
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    loads = [rows + (37 if e % 2 else -37) for e in range(E)]
    off = torch.tensor(loads, device=DEV).cumsum(0)
    L, dtype = sum(loads), torch.bfloat16
    X = torch.randn(L, K, generator=g, device=DEV).to(dtype)
    DY = torch.randn(L, N, generator=g, device=DEV).to(dtype)
    idx = torch.randperm(L, generator=g, device=DEV)
    DW, _ = ops.group_bwd_W(DY, X[idx], off, E)
    DWg, Db = ops.group_bwd_W(DY, X, off, E, has_bias=True, gather=(idx, 1))
    assert torch.equal(DW, DWg)
    lo = 0
    for e, n in enumerate(loads):
        x, y = X[idx[lo:lo + n]].double(), DY[lo:lo + n].double()
        _check(DW[e], x.t() @ y, x.abs().t() @ y.abs(), n, dtype)
        _check(Db[e], y.sum(0), y.abs().sum(0), n, dtype)
        lo += n


def test_unaligned_output():
    """An output two bytes off a 16-byte boundary takes the plain stores; the same bits."""
    g = torch.Generator(device=DEV).manual_seed(5)
    E, n, K, N = 4, 100, 136, 72
    off = torch.arange(1, E + 1, device=DEV) * n
    X = torch.randn(E * n, K, generator=g, device=DEV).bfloat16()
    DY = torch.randn(E * n, N, generator=g, device=DEV).bfloat16()
    DW, _ = ops.group_bwd_W(DY, X, off, E)
    buf = torch.zeros(E * N * K + 2, device=DEV, dtype=torch.bfloat16)
    out = buf[1:-1].view(E, N, K)
    ops._xty_launch(E, out.permute(0, 2, 1), None, DY, X, off)
    assert torch.equal(out.permute(0, 2, 1), DW) and buf[0] == 0 and buf[-1] == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gather_takes_any_index_vector(dtype):
    """`gather` stands for group() over the same index vector, also where that repeats rows and leaves others out."""
    g = torch.Generator(device=DEV).manual_seed(7)
    E, n, K, N, k = 4, 20, 136, 512, 2
    off = torch.arange(1, E + 1, device=DEV) * n
    X = torch.randn(E * n // k, K, generator=g, device=DEV).to(dtype)
    DY = torch.randn(E * n, N, generator=g, device=DEV).to(dtype)
    idx = torch.randint(0, E * n, (E * n,), generator=g, device=DEV)
    torch.full((E * n * K,), float("nan"), device=DEV, dtype=dtype)        # what a later allocation would find
    DW, Db = ops.group_bwd_W(DY, X, off, E, has_bias=True, gather=(idx, k))
    want, want_b = ops.group_bwd_W(DY, X[idx // k], off, E, has_bias=True)
    assert torch.equal(DW, want) and torch.equal(Db, want_b)


# dW on both sides of the lines between small and large tiles (output rows of whole 64-byte pieces or not, more than 512 tiles
# or not) and between lookups and a copy of the rows (N or K contiguous, wide or not): the same bits on every route
@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("E,rows,K,N", [(64, 90, 520, 2056), (64, 90, 544, 2080), (64, 100, 520, 2056), (16, 20, 1544, 6144),
                                        (64, 250, 768, 776), (4, 20, 264, 2056)])
def test_routes_of_few_rows(E, rows, K, N, layout):
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    loads = [rows + (7 if e % 2 else -7) for e in range(E)]
    off = torch.tensor(loads, device=DEV).cumsum(0)
    L, dtype = sum(loads), torch.bfloat16
    X = torch.randn(L // 2, K, generator=g, device=DEV).to(dtype)
    DY = torch.randn(L, N, generator=g, device=DEV).to(dtype)
    idx = torch.randperm(L, generator=g, device=DEV)
    like = torch.empty(E, K, N, dtype=dtype, device=DEV) if layout == "kn" else None
    DW, Db = ops.group_bwd_W(DY, X[idx // 2], off, E, has_bias=True, like=like)
    DWg, Dbg = ops.group_bwd_W(DY, X, off, E, has_bias=True, like=like, gather=(idx, 2))
    assert torch.equal(DW, DWg) and torch.equal(Db, Dbg)
    lo = 0
    for e, n in enumerate(loads):
        x, y = X[idx[lo:lo + n] // 2].double(), DY[lo:lo + n].double()
        _check(DW[e], x.t() @ y, x.abs().t() @ y.abs(), n, dtype)
        _check(Db[e], y.sum(0), y.abs().sum(0), n, dtype)
        lo += n


@pytest.mark.parametrize("n,N,dtype", [(400, 512, torch.bfloat16), (20, 6400, torch.bfloat16), (400, 6400, torch.float16),
                                       (20, 512, torch.float32), (400, 512, torch.float32)])
@pytest.mark.parametrize("k", [2, 4])
def test_gather_takes_any_index_vector_on_every_route(n, N, dtype, k):
    """The same where the rows are looked up inside the launch (n = 400, N = 512) and where the launch declines lookups
    (dY beyond 6144 columns, float32)."""
    g = torch.Generator(device=DEV).manual_seed(n + N)
    E, K = 4, 136
    off = torch.arange(1, E + 1, device=DEV) * n
    X = torch.randn(E * n // k, K, generator=g, device=DEV).to(dtype)
    DY = torch.randn(E * n, N, generator=g, device=DEV).to(dtype)
    idx = torch.randint(0, E * n, (E * n,), generator=g, device=DEV)
    torch.full((E * n * K,), float("nan"), device=DEV, dtype=dtype)
    DW, Db = ops.group_bwd_W(DY, X, off, E, has_bias=True, gather=(idx, k))
    want, want_b = ops.group_bwd_W(DY, X[idx // k], off, E, has_bias=True)
    assert torch.equal(DW, want) and torch.equal(Db, want_b)
