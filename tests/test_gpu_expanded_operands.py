"""Operands whose rows lie on top of each other (an expanded row): the same result as of a copy, in every form of the kernels."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows", [300, 2048])              # 256 x 128 tiles and the form of many rows
@pytest.mark.parametrize("which", ["DY", "X"])
def test_weight_gradient(rows, which):
    g = torch.Generator(device=DEV).manual_seed(rows)
    E, K, N = 2, 2568, 2824
    off = torch.tensor([rows - 7, 2 * rows], device=DEV)
    t = {"DY": torch.randn(2 * rows, N, generator=g, device=DEV).bfloat16(),
         "X": torch.randn(2 * rows, K, generator=g, device=DEV).bfloat16()}
    t[which] = t[which][:1].expand(2 * rows, -1)
    c = {n: v.contiguous() for n, v in t.items()}
    a, _ = ops.group_bwd_W(t["DY"], t["X"], off, E)
    b, _ = ops.group_bwd_W(c["DY"], c["X"], off, E)
    assert torch.equal(a, b)


@pytest.mark.parametrize("K", [1024, 2048])
def test_weights(K):
    """W[e] of one row, expanded over the contraction."""
    g = torch.Generator(device=DEV).manual_seed(K)
    E, k, T, N = 2, 1, 1200, 14336
    X = torch.randn(T, K, generator=g, device=DEV).bfloat16()
    W = torch.randn(E, 1, N, generator=g, device=DEV).bfloat16().expand(E, K, N)
    experts = torch.randint(0, E, (T, k), generator=g, device=DEV)
    eid, idx, off = ops.route(experts, E)
    a = ops.scatter2scatter(X, W, eid, idx, k, expert_offsets=off)
    b = ops.scatter2scatter(X, W.contiguous(), eid, idx, k, expert_offsets=off)
    assert torch.equal(a, b)
