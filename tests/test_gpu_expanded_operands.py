"""Operands whose rows lie on top of each other (an expanded row): the same result as of a copy, in every form of the kernels."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# Shapes whose copies go in 256 x 128 tiles (300 rows) and in the form of many rows (2048): see test_dispatch_lines, which asks the
# rules; 264 tiles of 256 x 256 leave the chip idle in a second round and go in small tiles, which take any rows
@pytest.mark.parametrize("E,K,N", [(4, 2056, 1544), (2, 2568, 2824)])
@pytest.mark.parametrize("rows", [300, 2048])
@pytest.mark.parametrize("which", ["DY", "X"])
def test_weight_gradient(rows, which, E, K, N):
    g = torch.Generator(device=DEV).manual_seed(rows)
    L = E * rows
    off = torch.tensor([rows - 7, 2 * rows, 3 * rows + 1, L][:E - 1] + [L], device=DEV)
    t = {"DY": torch.randn(L, N, generator=g, device=DEV).bfloat16(),
         "X": torch.randn(L, K, generator=g, device=DEV).bfloat16()}
    t[which] = t[which][:1].expand(L, -1)
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
