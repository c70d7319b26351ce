"""scatter2scatter around the line between 256 x 128 and 256 x 256 tiles (tile rows expected for even loads times columns of
128 at most 256): the last column count below it and the first above, even and uneven loads, both weight layouts, plain and
with each half of the gated unit.  Every row against a float32 product per expert."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16

#        E, rows, N: 25 tile rows x 10 columns and 12; 24 x 10 and 11; 3 x 3; 64 x 4 and 5
CASES = [(4, 1500, 1280), (4, 1500, 1416), (8, 600, 1160), (8, 600, 1288), (3, 240, 264), (32, 440, 392), (32, 440, 520)]


@pytest.mark.parametrize("skew", [0.0, 0.8])
@pytest.mark.parametrize("n_contig", [False, True])
@pytest.mark.parametrize("E,rows,N", CASES)
def test_both_sides(E, rows, N, n_contig, skew):
    g = torch.Generator(device=DEV).manual_seed(N)
    K, w = 200, [1.0 / (1 + e) ** skew for e in range(E)]
    loads = [int(rows * E * v / sum(w)) for v in w]
    L = sum(loads)
    experts = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(loads, device=DEV))
    experts = experts[torch.randperm(L, generator=g, device=DEV)].view(L, 1)
    eid, idx, off = ops.route(experts, E)
    X = torch.randn(L, K, generator=g, device=DEV).to(BF)
    W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.1).to(BF).permute(0, 2, 1)
    W = W.contiguous() if n_contig else W
    out = torch.full((L, N), float("nan"), dtype=BF, device=DEV)
    ops.scatter2scatter(X, W, eid, idx, 1, expert_offsets=off, out=out)
    lo = 0
    for e, n in enumerate(loads):
        r = idx[lo:lo + n]
        x, w_ = X[r].float(), W[e].float()
        want, mass = x @ w_, x.abs() @ w_.abs()
        # one rounding to bfloat16; two float32 sums of K products in different orders
        assert bool(((out[r].float() - want).abs() <= 2.0 ** -8 * want.abs() + 2 * K * 2.0 ** -24 * mass).all()), n
        lo += n
    pre, h = ops.scatter2scatter_glu(X, W, eid, idx, 1, expert_offsets=off)
    assert torch.equal(pre, out[idx])
    ref = ops.glu_fwd(pre)
    assert bool(((h.float() - ref.float()).abs() <= 2 ** -7 * ref.float().abs() + 1e-30).all())
    saved = torch.randn(L, 2 * N, generator=g, device=DEV).to(BF)
    dpre = ops.scatter2scatter_glu_bwd(X, W, saved, eid, idx, expert_offsets=off)      # rows in grouped order
    dh = ops.scatter2scatter(X, W, eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off)
    ref = ops.glu_bwd(saved, dh)
    assert bool(((dpre.float() - ref.float()).abs() <= 2 ** -7 * ref.float().abs() + 1e-30).all())
