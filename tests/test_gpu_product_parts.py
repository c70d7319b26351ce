"""Products of few tiles and a long contraction, whose contraction is cut into parts (whole_parts_for in csrc/gemm_mfma.hpp):
edges of tiles and columns, parts of unequal length, experts without rows, rows without an expert."""
import pytest
import torch

from scattermoe_amd import _C
from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("w_layout", ["k_contig", "n_contig"])
@pytest.mark.parametrize("loads,dropped,K,N,parts", [
    ([130], 0, 4480, 264, 8),                # 70 slices: seven parts of nine, one of seven
    ([257, 0, 300, 64], 9, 3648, 512, None),      # no rows, a second tile row of one row, rows that belong to no expert
    ([112, 113, 193, 255, 256, 1, 240, 50], 0, 14336, 1000, None)])
def test_whole_products_in_contraction_parts(loads, dropped, K, N, parts, w_layout, dtype):
    E, L = len(loads), sum(loads) + dropped
    g = torch.Generator(device=DEV).manual_seed(L)
    X = torch.randn(L, K, generator=g, device=DEV).to(dtype)
    W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.03).to(dtype).permute(0, 2, 1)
    W = W.contiguous() if w_layout == "n_contig" else W
    b = torch.randn(E, N, generator=g, device=DEV).to(dtype)
    off = torch.tensor(loads, device=DEV).cumsum(0)
    eid = torch.repeat_interleave(torch.arange(E + 1, device=DEV), torch.tensor(loads + [dropped], device=DEV))
    idx = torch.randperm(L, generator=g, device=DEV)
    need = _C.load().smoe_scatter2scatter_workspace_bytes(L, K, N, E, _C.float_code(dtype))
    assert need > 0 and need % (4 * L * N) == 0 and (parts is None or need == 4 * L * N * parts), need / (4 * L * N)
    for bias, x_grouped, y_grouped in ((b, True, False), (None, False, True), (b, True, True)):
        run = lambda: ops.scatter2scatter(X, W, eid, idx, 1, b=bias, x_grouped=x_grouped, y_grouped=y_grouped,
                                          out=torch.full((L, N), 7.0, device=DEV, dtype=dtype), expert_offsets=off)
        got, lo = run(), 0
        assert torch.equal(got, run())
        for e, n in enumerate(loads):
            src, dst = (torch.arange(lo, lo + n, device=DEV) if grouped else idx[lo:lo + n] for grouped in (x_grouped, y_grouped))
            x, w = X[src].double(), W[e].double()
            want = x @ w + (0.0 if bias is None else bias[e].double())
            # one rounding to the 16-bit type, and at most K float32 roundings of partial sums below the sum of magnitudes
            bound = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * want.abs() + K * 2.0 ** -24 * (x.abs() @ w.abs()) + 1e-6
            assert bool(((got[dst].double() - want).abs() <= bound).all()), (e, n)
            lo += n
        rest = torch.arange(lo, L, device=DEV) if y_grouped else idx[lo:]
        assert bool((got[rest] == 7.0).all())                 # rows without an expert are written by nobody
