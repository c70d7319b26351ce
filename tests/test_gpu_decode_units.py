"""Layer 2 of the two-launch decode step spreads (tile of rows, share of the contraction) units over the waves of a
workgroup: unit counts below, at and above the wave counts of both kernels (8 and 16), shares 1 to 4, tiles of 1, 2
and 4 rows - bit for bit against the general path."""
import pytest
import torch

from scattermoe_amd.kernels import ops
from test_gpu_decode_fused import _general

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("experts", [[[9, 3, 14, 0, 7, 11, 2, 5]], [[4, 4, 4, 4, 4, 4, 4, 4]], [[1, 2], [2, 1], [3, 1], [1, 2]]])
@pytest.mark.parametrize("F", [8, 512, 520, 1536, 2056, 4104])
def test_decode_units(experts, F):
    experts = torch.tensor(experts, device=DEV)
    (T, k), E, d = experts.shape, 16, 136
    g = torch.Generator(device=DEV).manual_seed(F)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    x, p, w1, b1, w2, b2 = r(T, d), r(T, k), r(E, 2 * F, d) * 0.1, r(E, 2 * F), r(E, d, F) * 0.1, r(E, d)
    got = ops.decode_glu_mlp(x, p, experts, w1, b1, w2, b2)
    assert got is not None and torch.equal(got, _general(x, p, experts, w1, b1, w2, b2, ops.ACT_SILU, E))
