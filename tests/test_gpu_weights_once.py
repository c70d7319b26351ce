"""Products with few rows per expert and more weights than the memory-side cache holds: experts of one tile row read them with the
non-temporal hint (reads_weights_once in csrc/gemm_mfma.hpp), the others in the same launch do not."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOADS = [0, 1, 63, 64, 65, 128, 129, 192, 193, 255, 256, 257, 300, 512, 513, 0]      # every height, one tile row and more


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("w_layout", ["k_contig", "n_contig"])
@pytest.mark.parametrize("K,N", [(2048, 1416), (1024, 2752)])            # 256 x 256 tiles, paired ones; a last column of 136, 64
def test_products_that_read_weights_once(K, N, w_layout, dtype):
    loads, dropped = LOADS * 4, 5
    E, L = len(loads), sum(loads) + dropped
    assert E * K * N * 2 >= 320 << 20 and 112 <= L // E < 640
    g = torch.Generator(device=DEV).manual_seed(K)
    X = torch.randn(L, K, generator=g, device=DEV).to(dtype)
    W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.03).to(dtype).permute(0, 2, 1)
    W = W.contiguous() if w_layout == "n_contig" else W
    off = torch.tensor(loads, device=DEV).cumsum(0)
    eid = torch.repeat_interleave(torch.arange(E + 1, device=DEV), torch.tensor(loads + [dropped], device=DEV))
    idx = torch.randperm(L, generator=g, device=DEV)
    got = ops.scatter2scatter(X, W, eid, idx, 1, y_grouped=True, out=torch.full((L, N), 7.0, device=DEV, dtype=dtype),
                              expert_offsets=off)
    lo = 0
    for e, n in enumerate(loads):
        x, w = X[idx[lo:lo + n]].float(), W[e].float()
        want = x @ w
        # one rounding to the 16-bit type, and at most K float32 roundings on either side below the sum of magnitudes
        bound = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * want.abs() + 2 * K * 2.0 ** -24 * (x.abs() @ w.abs()) + 1e-6
        assert bool(((got[lo:lo + n].float() - want).abs() <= bound).all()), (e, n)
        lo += n
    assert bool((got[lo:] == 7.0).all())                                  # rows without an expert are written by nobody
