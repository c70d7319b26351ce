"""Routing at the edges of its paths: rows per wave and per workgroup (256, 1024, 4096, 16384 and one more or less), one
to several chunks, expert counts around the 64 of a scan step and the 512 of the 16-wave workgroups; ids that are no
expert are left out."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("E", [1, 8, 63, 65, 128, 512, 513, 2048])
@pytest.mark.parametrize("L", [1, 63, 65, 256, 257, 1025, 4096, 4097, 16384, 16385, 270000])
def test_stable_sort_by_expert(L, E):
    g = torch.Generator(device=DEV).manual_seed(L + E)
    ids = (torch.rand(L, generator=g, device=DEV) ** 3 * E).long().clamp(max=E - 1)
    eid, idx, off = ops.route(ids, E)
    s_eid, s_idx = torch.sort(ids, stable=True)
    assert torch.equal(eid, s_eid) and torch.equal(idx, s_idx)
    assert torch.equal(off, torch.bincount(ids, minlength=E).cumsum(0))


@pytest.mark.parametrize("L", [200, 3000, 9000, 40000])
def test_ids_that_are_no_expert(L):
    E = 40
    ids = torch.randint(-3, E + 3, (L,), generator=torch.Generator().manual_seed(L)).to(DEV)
    eid, idx, off = ops.route(ids, E)
    rows = torch.nonzero((ids >= 0) & (ids < E)).flatten()
    s_eid, order = torch.sort(ids[rows], stable=True)
    assert torch.equal(eid[:len(rows)], s_eid) and torch.equal(idx[:len(rows)], rows[order])
    assert torch.equal(off, torch.bincount(ids[rows], minlength=E).cumsum(0))
