"""Launches whose tiles are taken in chunks per XCD (experts with equally many tile rows) and the choice against the other
order: one to three groups of 64 experts, one and several chunks per XCD, fewer tiles than XCDs, experts without rows,
loads on both sides of "a quarter apart".  Every row against a float32 product per expert; rows left out show as NaN."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV, BF = "cuda:0", torch.bfloat16


def _loads(kind, E, rows):
    if kind == "even":
        return [rows - (e * 7) % 5 for e in range(E)]
    if kind == "gaps":                       # a third of the experts has no rows
        return [0 if e % 3 == 1 else rows - e % 4 for e in range(E)]
    if kind == "one_more":                   # the last expert: another tile row
        return [rows] * (E - 1) + [rows + 256]
    if kind in ("first_low", "first_high"):  # three and four tile rows of 256: even, whichever comes first
        low = [E // 2] if kind == "first_high" else [0]
        return [3 * 256 - 5 if e in low else 4 * 256 - e % 9 for e in range(E)]
    if kind == "heights":                    # one tile row of 256 each, a few rows to all of them
        return [60 + (190 * e) // (E - 1) for e in range(E)]
    if kind == "heights_gaps":               # the same, every fourth expert without rows, loads falling
        return [0 if e % 4 == 2 else 250 - (190 * e) // (E - 1) for e in range(E)]
    if kind == "blocks":                     # a multiple of 256 between them: another tile row, another block of 64
        return [rows // 256 * 256 - e % 5 + (20 if e % 3 == 0 else 0) for e in range(E)]
    if kind == "blocks_gaps":                # the same, the last expert without rows
        return [0 if e == E - 1 else rows // 256 * 256 - e % 5 + (20 if e == 0 else 0) for e in range(E)]
    if kind == "tile_rows_gaps":             # two tile rows each, the first and every third expert without rows
        return [0 if e % 3 == 0 else rows - e % 4 for e in range(E)]
    return [rows * 4] + [max(1, rows // 8)] * (E - 1)       # uneven


@pytest.mark.parametrize("kind", ["even", "gaps", "one_more", "uneven"])
@pytest.mark.parametrize("E,rows,K,N", [
    (32, 310, 264, 2568),      # two tile rows of 256, three rounds: several chunks
    (3, 1300, 1856, 648),      # six or seven tile rows, one wave per SIMD
    (65, 9, 2112, 1032),       # weight streams: one chunk, two groups of experts
    (130, 40, 256, 264), (9, 70, 512, 520), (2, 20, 1024, 64), (16, 130, 264, 2056),
])
@pytest.mark.parametrize("n_contig", [False, True])
def test_plain_and_gated(E, rows, K, N, n_contig, kind):
    _check_plain_and_gated(E, rows, K, N, n_contig, kind)


@pytest.mark.parametrize("kind", ["first_low", "first_high", "heights", "heights_gaps", "tile_rows_gaps", "blocks",
                                  "blocks_gaps"])
@pytest.mark.parametrize("E,rows,K,N", [(32, 500, 264, 2568), (66, 500, 264, 1032), (17, 500, 1856, 648),
                                        (130, 530, 264, 264), (64, 300, 264, 2056)])
@pytest.mark.parametrize("n_contig", [False, True])
def test_loads_at_the_rule(E, rows, K, N, n_contig, kind):
    """Loads that count as even whatever expert comes first, those whose tile rows agree while their heights do
    not, and those whose tile rows differ while their blocks of 64 rows hardly do."""
    _check_plain_and_gated(E, rows, K, N, n_contig, kind)


def _check_plain_and_gated(E, rows, K, N, n_contig, kind):
    g = torch.Generator(device=DEV).manual_seed(E + rows)
    loads = _loads(kind, E, rows)
    L = sum(loads)
    experts = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(loads, device=DEV))
    experts = experts[torch.randperm(L, generator=g, device=DEV)].view(L, 1)
    eid, idx, off = ops.route(experts, E)
    X = torch.randn(L, K, generator=g, device=DEV).to(BF)
    W = (torch.randn(E, N, K, generator=g, device=DEV) * 0.1).to(BF).permute(0, 2, 1)
    W = W.contiguous() if n_contig else W
    out = torch.full((L, N), float("nan"), dtype=BF, device=DEV)
    ops.scatter2scatter(X, W, eid, idx, 1, expert_offsets=off, out=out)
    ends = [0] + off.tolist()
    for e in range(E):
        r = idx[ends[e]:ends[e + 1]]
        x, w = X[r].float(), W[e].float()
        want, mass = x @ w, x.abs() @ w.abs()
        # one rounding to bfloat16; two float32 sums of K products in different orders
        assert bool(((out[r].float() - want).abs() <= 2.0 ** -8 * want.abs() + 2 * K * 2.0 ** -24 * mass).all()), loads[e]
    pre, h = ops.scatter2scatter_glu(X, W, eid, idx, 1, expert_offsets=off)
    assert torch.equal(pre, out[idx])
    ref = ops.glu_fwd(pre)
    assert bool(((h.float() - ref.float()).abs() <= 2 ** -7 * ref.float().abs() + 1e-30).all())
