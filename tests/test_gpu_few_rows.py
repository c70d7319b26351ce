"""scatter2scatter with fewer than 52 rows per expert: one case per branch of the tile choice (expected workgroups of
128-wide tiles below 192, below 256, from 256, between 512 and 768, beyond; column counts that do and do not divide
among 8 XCDs; rows per expert below 16, below 24, from 24, on both sides of 64 minus three standard deviations), both
weight layouts, plain and with the gated unit, a contraction that is no multiple of 64, uneven loads. Against a
float32 product per expert on the same values; bar rel 2e-2 / abs 1e-2 scaled by the magnitude a dot product of that
length reaches (as in test_gpu_random_shapes)."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16

#        E   avg  K    N
CASES = [(48, 4, 200, 1408), (48, 40, 72, 1408), (16, 6, 264, 2048), (8, 5, 264, 1024), (8, 30, 264, 1000),
         (96, 5, 136, 1536), (96, 30, 136, 1536), (128, 9, 520, 1024), (100, 20, 64, 1032),
         (48, 44, 136, 1928), (48, 45, 136, 1928)]


@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("n_contig", [False, True])
@pytest.mark.parametrize("E,avg,K,N", CASES)
def test_few_rows(E, avg, K, N, n_contig, glu):
    g = torch.Generator(device=DEV).manual_seed(E + avg + K)
    T = E * avg // 2
    logits = torch.randn(T, E, generator=g, device=DEV) - torch.linspace(0, 1.5, E, device=DEV)
    experts = torch.topk(logits, 2).indices
    eid, idx, off = ops.route(experts, E)
    X = torch.randn(T, K, generator=g, device=DEV).to(BF)
    W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.1).to(BF).permute(0, 2, 1)
    b = torch.randn(E, N, generator=g, device=DEV).to(BF)
    Wd = W.contiguous() if n_contig else W
    want = torch.empty(2 * T, N, device=DEV)
    ends = [0] + off.tolist()
    for e in range(E):
        rows = slice(ends[e], ends[e + 1])
        want[rows] = X[idx[rows] // 2].float() @ W[e].float() + b[e].float()
    if glu:
        pre, h = ops.scatter2scatter_glu(X, Wd, eid, idx, 2, b=b, expert_offsets=off)
        first, second = pre.float().chunk(2, -1)
        torch.testing.assert_close(h.float(), torch.nn.functional.silu(second) * first, rtol=2e-2, atol=1e-2)
        got = pre
    else:
        got = ops.scatter2scatter(X, Wd, eid, idx, 2, b=b, y_grouped=True, expert_offsets=off)
        slots = ops.scatter2scatter(X, Wd, eid, idx, 2, b=b, expert_offsets=off)
        assert torch.equal(slots[idx], got)
    err = (got.float() - want).abs()
    assert bool((err <= 1e-2 * (0.1 * K ** 0.5 + 1) + 2e-2 * want.abs()).all()), float(err.max())
