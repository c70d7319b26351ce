"""256 x 256 tiles are multiplied at the height of their rows (1 to 4 blocks of 64): expert loads on both sides of every
multiple of 64 up to two tiles (mean above 224: always this class), both forms of the class (contraction of 1856: one wave per SIMD, of 264: eight waves),
both weight layouts, plain and with every fused unit.  Plain products against a float32 product per expert (rel 2e-2 /
abs 1e-2 scaled by the magnitude of the dot products); fused ones against the unfused launches of the same product,
whose intermediate they round at the same point (one unit in the last place of bfloat16 for the unit's own result)."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16
LOADS = [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 321, 449, 0, 512, 513, 700]


def _problem(K, N, n_contig, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    E, L = len(LOADS), sum(LOADS)
    experts = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(LOADS, device=DEV))
    experts = experts[torch.randperm(L, generator=g, device=DEV)].view(L, 1)
    eid, idx, off = ops.route(experts, E)
    X = torch.randn(L, K, generator=g, device=DEV).to(BF)
    W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.1).to(BF).permute(0, 2, 1)
    return g, E, L, eid, idx, off, X, (W.contiguous() if n_contig else W)


@pytest.mark.parametrize("n_contig", [False, True])
@pytest.mark.parametrize("K,N", [(1856, 2320), (264, 2568)])
def test_plain(K, N, n_contig):
    g, E, L, eid, idx, off, X, W = _problem(K, N, n_contig, 1)
    b = torch.randn(E, N, generator=g, device=DEV).to(BF)
    out = torch.full((L, N), float("nan"), dtype=BF, device=DEV)
    ops.scatter2scatter(X, W, eid, idx, 1, b=b, expert_offsets=off, out=out)
    ends = [0] + off.tolist()
    for e in range(E):
        rows = idx[ends[e]:ends[e + 1]]
        want = X[rows].float() @ W[e].float() + b[e].float()
        err = (out[rows].float() - want).abs()
        assert bool((err <= 1e-2 * (0.1 * K ** 0.5 + 1) + 2e-2 * want.abs()).all()), (LOADS[e], float(err.max()))


@pytest.mark.parametrize("n_contig", [False, True])
@pytest.mark.parametrize("K,F", [(1856, 1288), (264, 1288)])
@pytest.mark.parametrize("act", [ops.ACT_SILU, ops.ACT_SILU_GATE_FIRST, ops.ACT_GPT_OSS])
def test_fused(act, K, F, n_contig):
    g, E, L, eid, idx, off, X, W1 = _problem(K, 2 * F, n_contig, 2)
    pre, h = ops.scatter2scatter_glu(X, W1, eid, idx, 1, act=act, expert_offsets=off)
    assert torch.equal(pre, ops.scatter2scatter(X, W1, eid, idx, 1, y_grouped=True, expert_offsets=off))
    ref = ops.gpt_oss_glu(pre) if act == ops.ACT_GPT_OSS else ops.glu_fwd(pre, act)
    assert bool(((h.float() - ref.float()).abs() <= 2 ** -7 * ref.float().abs() + 1e-30).all())
    W2 = (torch.randn(E, F, K, generator=g, device=DEV) * 0.1).to(BF).permute(0, 2, 1)       # (E, K, F): dY @ W2
    W2 = W2.contiguous() if n_contig else W2
    dpre = ops.scatter2scatter_glu_bwd(X, W2, pre, eid, idx, act=act, expert_offsets=off)
    dh = ops.scatter2scatter(X, W2, eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off)
    if act == ops.ACT_GPT_OSS:
        leaf = pre.clone().requires_grad_()
        (ref,) = torch.autograd.grad(ops.gpt_oss_glu(leaf), leaf, dh)
    else:
        ref = ops.glu_bwd(pre, dh, act)
    assert bool(((dpre.float() - ref.float()).abs() <= 2 ** -7 * ref.float().abs() + 1e-30).all())
