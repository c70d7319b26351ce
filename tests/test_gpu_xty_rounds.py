"""Weight gradients of 1280 to 2047 rows per expert and four rounds of 256 x 256 tiles, which the one-wave-per-SIMD form takes
(xty_one_wave in csrc/gemm_mfma.hpp): remainders of rows and columns, an expert without rows, rows that belong to no expert."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n_contig", [False, True])
def test_weight_gradients_of_four_rounds(n_contig, dtype):
    loads, dropped, N, K = [1280, 0, 1, 65, 2047, 1344, 2600, 2905], 5, 2824, 2696
    E, L = len(loads), sum(loads) + dropped
    assert 1280 <= L // E < 2048 and E * ((N + 255) // 256) * ((K + 255) // 256) >= 1024
    g = torch.Generator(device=DEV).manual_seed(L)
    DY = torch.randn(L, N, generator=g, device=DEV).to(dtype)
    X = torch.randn(L, K, generator=g, device=DEV).to(dtype)
    off = torch.tensor(loads, device=DEV).cumsum(0)
    DW, _ = ops.group_bwd_W(DY, X, off, E, like=torch.empty(E, K, N, device="meta") if n_contig else None)
    lo = 0
    for e, n in enumerate(loads):
        x, dy = X[lo:lo + n].float(), DY[lo:lo + n].float()
        want, size = x.t().contiguous() @ dy, x.abs().t().contiguous() @ dy.abs()
        # one rounding to the 16-bit type, and at most n float32 roundings on either side below the sum of magnitudes
        bound = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * want.abs() + 2 * n * 2.0 ** -24 * size + 1e-6
        assert bool(((DW[e].float() - want).abs() <= bound).all()), (e, n)
        lo += n
