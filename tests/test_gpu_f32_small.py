"""float32 launches of few tiles, in 32 x 32 tiles of a quarter of the contraction per wave: expert loads and output columns on
both sides of a tile's edge, contractions shorter than one wave's chunk, of a partial last one, and of several steps per wave;
both weight layouts, gathered and grouped rows, both layouts of the weight gradient, bias.  Against float64: a float32 sum
of n products of total magnitude `mass` in any order is off by at most n 2^-24 mass, one more rounding for the bias."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOADS = [1, 31, 32, 33, 0, 64, 65, 6, 0, 4]          # 236 rows, 10 experts


def _check(got, want, mass, n):
    assert bool(((got.double() - want).abs() <= (n + 2) * 2.0 ** -24 * mass + 1e-30).all())


def _inputs(K, N, k, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + K + N)
    E, L = len(LOADS), sum(LOADS)
    experts = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(LOADS, device=DEV))
    experts = experts[torch.randperm(L, generator=g, device=DEV)].view(L // k, k)
    eid, idx, off = ops.route(experts, E)
    X = torch.randn(L // k, K, generator=g, device=DEV)
    W = torch.randn(E, N, K, generator=g, device=DEV).permute(0, 2, 1)
    b = torch.randn(E, N, generator=g, device=DEV)
    return g, E, L, eid, idx, off, X, W, b


@pytest.mark.parametrize("n_contig", [False, True])
@pytest.mark.parametrize("K,N", [(4, 4), (28, 36), (32, 32), (36, 64), (100, 100), (132, 28), (260, 96), (600, 132), (1, 1), (3, 5), (35, 66), (101, 133), (682, 31)])
def test_products(K, N, n_contig):
    g, E, L, eid, idx, off, X, W, b = _inputs(K, N, 4)
    W = W.contiguous() if n_contig else W
    grouped = ops.scatter2scatter(X, W, eid, idx, 4, b=b, y_grouped=True, expert_offsets=off)
    out = torch.full((L, N), float("nan"), device=DEV)
    ops.scatter2scatter(X[idx // 4], W, eid, idx, 1, b=b, x_grouped=True, expert_offsets=off, out=out)
    assert torch.equal(out[idx], grouped)
    lo = 0
    for e, hi in enumerate(off.tolist()):
        x, w = X[idx[lo:hi] // 4].double(), W[e].double()
        _check(grouped[lo:hi], x @ w + b[e].double(), x.abs() @ w.abs() + b[e].double().abs(), K)
        lo = hi


@pytest.mark.parametrize("layout", ["nk", "kn"])
@pytest.mark.parametrize("K,N", [(4, 36), (32, 32), (100, 132), (128, 256), (1, 3), (33, 35), (101, 682)])
def test_weight_gradients(K, N, layout):
    g, E, L, eid, idx, off, X, W, b = _inputs(K, N, 1)
    DY = torch.randn(L, N, generator=g, device=DEV)
    like = torch.empty(E, K, N, device=DEV) if layout == "kn" else None
    DW, Db = ops.group_bwd_W(DY, X, off, E, has_bias=True, like=like)
    lo = 0
    for e, hi in enumerate(off.tolist()):
        x, y = X[lo:hi].double(), DY[lo:hi].double()
        _check(DW[e], x.t() @ y, x.abs().t() @ y.abs(), hi - lo)
        _check(Db[e], y.sum(0), y.abs().sum(0), hi - lo)
        lo = hi


def test_unaligned_operands():
    """Operands and outputs that begin one element into wider matrices; more tiles than the aligned ones may have."""
    for K, N in ((68, 3300), (67, 3301), (131, 3301)):      # 182 tiles of 128 x 128: the last goes in 32 x 32 ones
        g, E, L, eid, idx, off, X, W, b = _inputs(K + 1, N + 1, 1)
        X, W = X[:, 1:], W[:, 1:, 1:]
        DY = torch.randn(L, N + 1, generator=g, device=DEV)[:, 1:]
        out = torch.full((L, N + 1), 7.0, device=DEV)
        ops.scatter2scatter(X, W, eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off, out=out[:, 1:])
        dx = ops.scatter2scatter(DY, W.permute(0, 2, 1), eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off)
        DW, Db = ops.group_bwd_W(DY, X, off, E, has_bias=True)
        assert bool((out[:, 0] == 7.0).all())
        lo = 0
        for e, hi in enumerate(off.tolist()):
            x, w, y = X[lo:hi].double(), W[e].double(), DY[lo:hi].double()
            _check(out[lo:hi, 1:], x @ w, x.abs() @ w.abs(), K)
            _check(dx[lo:hi], y @ w.t(), y.abs() @ w.t().abs(), N)
            _check(DW[e], x.t() @ y, x.abs().t() @ y.abs(), hi - lo)
            _check(Db[e], y.sum(0), y.abs().sum(0), hi - lo)
            lo = hi


def test_infinities_stay_with_their_rows():
    """Neither a row beyond an expert's last one nor a contraction element beyond the last is multiplied, not even by zero."""
    g, E, L, eid, idx, off, X, W, b = _inputs(36, 64, 1)
    DY = torch.randn(L, 64, generator=g, device=DEV)
    want = ops.scatter2scatter(X, W, eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off)
    want_dw, _ = ops.group_bwd_W(DY, X, off, E)
    lo, hi = off[2].item(), off[3].item()
    bad_x, bad_dy = X.clone(), DY.clone()
    bad_x[lo:hi], bad_dy[lo:hi] = float("inf"), float("nan")
    got = ops.scatter2scatter(bad_x, W, eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off)
    dw, _ = ops.group_bwd_W(bad_dy, bad_x, off, E)
    rows = [r for r in range(L) if not lo <= r < hi]
    experts = [e for e in range(E) if e != 3]
    assert torch.equal(got[rows], want[rows]) and torch.equal(dw[experts], want_dw[experts])
    assert not bool(got[lo:hi].isfinite().any()) and bool(dw[3].isnan().all())
