"""Products of short contractions (whole 64-deep slices, fewer than 1792) in 256 x 128 tiles, two workgroups per CU: one slice,
two, an odd number and the longest; expert loads on both sides of every tile height; partly filled tile columns; both weight
layouts; plain against a float32 product per expert, fused units against the unfused launches (bounds of test_gpu_tile_heights);
gathered rows, whose table lies where operands are to come; and the same bits as the general form of the product."""
import pytest
import torch

from scattermoe_amd.kernels import ops
from test_gpu_tile_heights import BF, DEV, LOADS, _problem, test_fused as check_fused, test_plain as check_plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_contig", [False, True])
@pytest.mark.parametrize("K,N", [(64, 4104), (128, 2176), (576, 2312), (1728, 2400)])
def test_plain(K, N, n_contig):
    check_plain(K, N, n_contig)


@pytest.mark.parametrize("n_contig", [False, True])
@pytest.mark.parametrize("act", [ops.ACT_SILU, ops.ACT_SILU_GATE_FIRST, ops.ACT_GPT_OSS])
@pytest.mark.parametrize("K,F", [(64, 2056), (320, 1544)])
def test_fused(act, K, F, n_contig):
    check_fused(act, K, F, n_contig)


@pytest.mark.parametrize("K,N", [(64, 4096), (704, 2176)])
def test_gathered_rows(K, N):
    g, E, L, eid, idx, off, X, W = _problem(K, N, False, 3)
    k = 4
    assert L % k == 0
    x = X[:L // k].contiguous()
    got = ops.scatter2scatter(x, W, eid, idx, k, expert_offsets=off, y_grouped=True)
    assert torch.equal(got, ops.scatter2scatter(x[idx // k], W, eid, idx, 1, x_grouped=True, y_grouped=True, expert_offsets=off))


@pytest.mark.parametrize("n_contig", [False, True])
def test_same_bits_as_unaligned_output(n_contig):
    """An output whose rows start between 16-byte pieces takes the eight-wave tiles: the same sums in the same order."""
    g, E, L, eid, idx, off, X, W = _problem(448, 2176, n_contig, 4)
    wide = torch.full((L, 2177), 7.0, dtype=BF, device=DEV)
    ops.scatter2scatter(X, W, eid, idx, 1, expert_offsets=off, out=wide[:, 1:])
    assert torch.equal(wide[:, 1:], ops.scatter2scatter(X, W, eid, idx, 1, expert_offsets=off))
    assert bool((wide[:, 0] == 7.0).all())


def test_uneven_loads_many_experts():
    """Loads that differ take the super tiles or column stripes instead of the chunks of neighbours."""
    for loads in ([6000, 40, 300, 0, 1, 2500, 64, 65], [17] * 60 + [9000] + [500] * 3):
        E, L, K, N = len(loads), sum(loads), 192, 1288
        g = torch.Generator(device=DEV).manual_seed(L)
        experts = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(loads, device=DEV)).view(L, 1)
        eid, idx, off = ops.route(experts, E)
        X = torch.randn(L, K, generator=g, device=DEV).to(BF)
        W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.1).to(BF).permute(0, 2, 1)
        out = torch.full((L, N), float("nan"), dtype=BF, device=DEV)
        ops.scatter2scatter(X, W, eid, idx, 1, expert_offsets=off, out=out)
        lo = 0
        for e, hi in enumerate(off.tolist()):
            want = X[lo:hi].float() @ W[e].float()
            assert bool(((out[lo:hi].float() - want).abs() <= 1e-2 * (0.1 * K ** 0.5 + 1) + 2e-2 * want.abs()).all())
            lo = hi
