"""Products of few rows per expert in tiles of 192 columns (narrow_columns in csrc/gemm_mfma.hpp): edges of tiles and columns, every
height, experts without rows and of more than one tile row; the gated units' gradients behind them."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOADS = [0, 1, 63, 64, 65, 128, 129, 192, 193, 255, 256, 257, 300, 0, 190, 240]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("w_layout", ["k_contig", "n_contig"])
@pytest.mark.parametrize("N", [2880, 2696, 2872])                 # a last column of 192, 8, 184; one and a half rounds of 256
def test_products_in_tiles_of_192_columns(N, w_layout, dtype):
    loads, dropped, K = LOADS * 2, 5, 1792
    E, L = len(loads), sum(loads) + dropped
    assert 112 <= L // E < 224
    g = torch.Generator(device=DEV).manual_seed(N)
    X = torch.randn(L, K, generator=g, device=DEV).to(dtype)
    W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.03).to(dtype).permute(0, 2, 1)
    W = W.contiguous() if w_layout == "n_contig" else W
    b = torch.randn(E, N, generator=g, device=DEV).to(dtype)
    off = torch.tensor(loads, device=DEV).cumsum(0)
    eid = torch.repeat_interleave(torch.arange(E + 1, device=DEV), torch.tensor(loads + [dropped], device=DEV))
    idx = torch.randperm(L, generator=g, device=DEV)
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for bias, x_grouped, y_grouped in ((b, True, False), (None, False, True), (None, True, True)):
        got = ops.scatter2scatter(X, W, eid, idx, 1, b=bias, x_grouped=x_grouped, y_grouped=y_grouped,
                                  out=torch.full((L, N), 7.0, device=DEV, dtype=dtype), expert_offsets=off)
        lo = 0
        for e, n in enumerate(loads):
            src, dst = (torch.arange(lo, lo + n, device=DEV) if grouped else idx[lo:lo + n] for grouped in (x_grouped, y_grouped))
            x, w = X[src].float(), W[e].float()
            want = x @ w + (0.0 if bias is None else bias[e].float())
            # one rounding to the 16-bit type, and at most K float32 roundings on either side below the sum of magnitudes
            bound = eps * want.abs() + 2 * K * 2.0 ** -24 * (x.abs() @ w.abs()) + 1e-6
            assert bool(((got[dst].float() - want).abs() <= bound).all()), (e, n)
            lo += n
        rest = torch.arange(lo, L, device=DEV) if y_grouped else idx[lo:]
        assert bool((got[rest] == 7.0).all())                     # rows without an expert are written by nobody
    # the units' gradients against the passes over the plain product: the same arithmetic, up to one unit in the last place
    pre = torch.randn(L, 2 * N, generator=g, device=DEV).to(dtype)
    dh, rows = got, slice(0, sum(loads))
    leaf = pre.clone().requires_grad_()
    ops.gpt_oss_glu(leaf).backward(dh)
    for act, want in ((ops.ACT_SILU, ops.glu_bwd(pre, dh)), (ops.ACT_GPT_OSS, leaf.grad)):
        dpre = ops.scatter2scatter_glu_bwd(X, W, pre, eid, idx, act=act, expert_offsets=off)
        bad = (dpre[rows].float() - want[rows].float()).abs() > 2 * eps * want[rows].float().abs() + 1e-6
        assert not bool(bad.any())
