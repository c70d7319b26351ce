"""Products with more weights than the memory-side cache holds in tiles of 256 columns, one wave per SIMD: experts of one tile row
read them with the non-temporal hint (reads_weights_once in csrc/gemm_mfma.hpp), the others in the same launch do not.  The
plain product, with every fused unit, and in contraction parts; that these are the classes is asserted in
test_dispatch_products."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOADS = [0, 1, 63, 64, 65, 128, 129, 192, 193, 255, 256, 257, 300, 512, 513, 0]      # every height, one tile row and more
K, N = 2048, 1680                                         # a last column of 144
PARTS = ([0, 64, 129, 193, 256, 257, 300, 200], 14336, 1536)


def _case(loads, K, N, w_layout, dtype):
    E, L = len(loads), sum(loads) + 5                     # (five rows that belong to no expert)
    g = torch.Generator(device=DEV).manual_seed(N)
    X = torch.randn(L, K, generator=g, device=DEV).to(dtype)
    W = (torch.randn(E, N, K, generator=g, device=DEV, dtype=dtype) * 0.03).permute(0, 2, 1)
    W = W.contiguous() if w_layout == "n_contig" else W
    off = torch.tensor(loads, device=DEV).cumsum(0)
    eid = torch.repeat_interleave(torch.arange(E + 1, device=DEV), torch.tensor(loads + [5], device=DEV))
    return X, W, eid, torch.randperm(L, generator=g, device=DEV), off, g


def _compare(got, X, W, idx, loads, dtype):
    """A product of gathered rows in grouped order against one in float64, expert by expert."""
    lo = 0
    for e, n in enumerate(loads):
        x, w = X[idx[lo:lo + n]].double(), W[e].double()
        want = x @ w
        # one rounding to the 16-bit type, and at most K float32 roundings below the sum of magnitudes
        bound = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * want.abs() + X.size(1) * 2.0 ** -24 * (x.abs() @ w.abs()) + 1e-6
        assert bool(((got[lo:lo + n].double() - want).abs() <= bound).all()), (e, n)
        lo += n
    return lo


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("w_layout", ["k_contig", "n_contig"])
def test_products_and_fused_units(w_layout, dtype):
    loads = LOADS * 4
    X, W, eid, idx, off, g = _case(loads, K, N, w_layout, dtype)
    L = X.size(0)
    assert W.numel() * 2 >= 320 << 20
    out = ops.scatter2scatter(X, W, eid, idx, 1, y_grouped=True, out=torch.full((L, N), 7.0, device=DEV, dtype=dtype),
                              expert_offsets=off)
    rows = _compare(out, X, W, idx, loads, dtype)
    assert bool((out[rows:] == 7.0).all())                # rows without an expert are written by nobody
    # the fused units against the passes over the plain product: the same arithmetic, up to one unit in the last place
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    close = lambda got, want: bool(((got[:rows].float() - want[:rows].float()).abs() <= 2 * eps * want[:rows].float().abs() + 1e-6).all())
    for act, unit in ((ops.ACT_SILU, ops.glu_fwd), (ops.ACT_GPT_OSS, ops.gpt_oss_glu)):
        pre, h = ops.scatter2scatter_glu(X, W, eid, idx, 1, act=act, expert_offsets=off)
        assert torch.equal(pre[:rows], out[:rows]) and close(h, unit(out)), act
    dh = ops.scatter2scatter(X, W, eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off)
    leaf = torch.randn(L, 2 * N, generator=g, device=DEV).to(dtype).requires_grad_()
    ops.gpt_oss_glu(leaf).backward(dh)
    pre = leaf.detach()
    for act, want in ((ops.ACT_SILU, ops.glu_bwd(pre, dh)), (ops.ACT_GPT_OSS, leaf.grad)):
        dpre = ops.scatter2scatter_glu_bwd(X, W, pre, eid, idx, act=act, expert_offsets=off)
        assert close(dpre, want), act


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("w_layout", ["k_contig", "n_contig"])
def test_contraction_parts(w_layout, dtype):
    loads, K, N = PARTS
    X, W, eid, idx, off, _ = _case(loads, K, N, w_layout, dtype)
    assert W.numel() * 2 >= 320 << 20
    out = ops.scatter2scatter(X, W, eid, idx, 1, y_grouped=True, out=torch.full((X.size(0), N), 7.0, device=DEV, dtype=dtype),
                              expert_offsets=off)
    assert bool((out[_compare(out, X, W, idx, loads, dtype):] == 7.0).all())
