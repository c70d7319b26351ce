"""Expert ids outside [0, E) (padding, sentinels): the routing drops their rows, and a training step has the weight
gradients of the rows that are kept, whatever the memory of the index vectors held before."""
import pytest
import torch

import scattermoe_amd as sm
from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ids(L, E, seed):
    g = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, E, (L,), generator=g)
    drop = torch.rand(L, generator=g) < 0.2
    return torch.where(drop, torch.tensor([-1, E, E + 5])[torch.randint(0, 3, (L,), generator=g)], ids).to(DEV), drop.to(DEV)


def _stale(L):
    """What a later allocation of L int64 would find: a slot that the routing places elsewhere."""
    torch.cuda.synchronize()
    [torch.zeros(L, dtype=torch.int64, device=DEV) for _ in range(4)]


@pytest.mark.parametrize("L,E", [(200, 40), (3000, 40), (3000, 600), (9000, 40), (40000, 40), (40000, 600), (600000, 8)])
def test_places_behind_the_last_row(L, E):
    ids, drop = _ids(L, E, L)
    _stale(L)
    eid, idx, off = ops.route(ids, E)
    n = int((~drop).sum())
    assert int(off[-1]) == n and bool((eid[n:] == E).all()) and bool((idx[n:] == -1).all())
    assert torch.equal(ops.offsets_from_sorted(eid, E), off)


@pytest.mark.parametrize("L", [7, 3000, 40000])
def test_ids_beyond_32_bits(L):
    """Their low half may look like an expert; the two-launch decode step (L = 7) and the routing agree on them."""
    E, d, F = 16, 64, 64
    ids = torch.arange(L, device=DEV) % E
    far = torch.arange(L, device=DEV) % 3 == 0
    wide = torch.where(far, ids + torch.where(ids % 2 == 0, 1 << 32, -(1 << 40)), ids)
    got, want = ops.route(wide, E), ops.route(torch.where(far, -1, ids), E)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    if L == 7:
        g = torch.Generator(device=DEV).manual_seed(1)
        r = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
        x, p, w1, w2 = r(1, d), r(1, L), r(E, 2 * F, d), r(E, d, F)
        a, b = (ops.decode_glu_mlp(x, p, e.view(1, L), w1, None, w2, None) for e in (wide, torch.where(far, -1, ids)))
        assert a is not None and torch.equal(a, b)


@pytest.mark.parametrize("dtype,K", [(torch.bfloat16, 136), (torch.bfloat16, 133), (torch.float32, 136)])
@pytest.mark.parametrize("coeff", [False, True])
def test_group_leaves_rows_without_a_slot(dtype, K, coeff):
    g = torch.Generator(device=DEV).manual_seed(K)
    L, k = 300, 2
    A = torch.randn(L // k, K, generator=g, device=DEV).to(dtype)
    c = torch.randn(L, generator=g, device=DEV).to(dtype) if coeff else None
    idx = torch.randperm(L, generator=g, device=DEV)
    none = torch.rand(L, generator=g, device=DEV) < 0.2
    out = torch.full((L, K), 7.0, device=DEV, dtype=dtype)
    got = ops.group(A, torch.where(none, torch.where(idx % 2 == 0, -1, L), idx), coeff=c, fan_out=k, out=out)
    want = A[idx // k].float() * (c[idx].float()[:, None] if coeff else 1.0)
    assert torch.equal(got[~none], want.to(dtype)[~none]) and bool((got[none] == 7.0).all())


# rows per expert on both sides of the copy in place of lookups, wide and narrow dY, float32, one slot per token
@pytest.mark.parametrize("T,k,N,dtype", [(200, 4, 1024, torch.bfloat16), (6000, 4, 1024, torch.float16),
                                         (200, 2, 6400, torch.bfloat16), (3000, 2, 6400, torch.bfloat16),
                                         (200, 2, 264, torch.float32), (400, 1, 1024, torch.bfloat16)])
def test_weight_gradient_over_the_kept_rows(T, k, N, dtype):
    g = torch.Generator(device=DEV).manual_seed(T + N)
    E, K, L = 8, 136, T * k
    ids, drop = _ids(L, E, T)
    _stale(L)
    eid, idx, off = ops.route(ids.view(T, k), E)
    n = int(off[-1])
    X = torch.randn(T, K, generator=g, device=DEV).to(dtype)
    DY = torch.randn(L, N, generator=g, device=DEV).to(dtype)
    rows = torch.zeros(L, K, device=DEV, dtype=dtype)
    rows[:n] = X[idx[:n] // k]
    want, want_b = ops.group_bwd_W(DY, rows, off, E, has_bias=True)
    got, got_b = ops.group_bwd_W(DY, X, off, E, has_bias=True, gather=(idx, k))
    assert torch.equal(got, want) and torch.equal(got_b, want_b)


@pytest.mark.parametrize("cls,T,k", [(sm.mlp.GLUMLP, 150, 4), (sm.mlp.GLUMLP, 3000, 2), (sm.mlp.MLP, 150, 4),
                                     (sm.mlp.MLP, 150, 1)])
def test_training_step_over_the_kept_rows(cls, T, k):
    """Against the step in which the dropped slots go to expert 0 with a gate of zero: they add exact zeros to the
    sums, so what differs is the order of float32 sums and their one rounding to bfloat16 (at most 2 x 2^-9 relative;
    near-cancelling sums of up to n terms: n 2^-24 of a mass that 1e-3 of the largest gradient covers by far)."""
    torch.manual_seed(T + k)
    E, d, F = 8, 136, 264
    kw = {} if cls is sm.mlp.GLUMLP else {"activation": torch.nn.GELU()}
    module = cls(d, F, E, k, bias=True, **kw).to(DEV, torch.bfloat16)
    ids, drop = _ids(T * k, E, T)
    ids, drop = ids.view(T, k), drop.view(T, k)
    gates = torch.rand(T, k, device=DEV).bfloat16()
    x, dy = torch.randn(T, d, device=DEV).bfloat16(), torch.randn(T, d, device=DEV).bfloat16()

    def grads(p, e):
        module.zero_grad()
        _stale(T * k)
        module(x, p, e).backward(dy)
        return [q.grad.float() for q in module.parameters()]

    want = grads(torch.where(drop, 0.0, gates).bfloat16(), torch.where(drop, 0, ids))
    for p in (gates, gates.clone().requires_grad_()):
        for got, ref in zip(grads(p, ids), want):
            assert bool(((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-3 * ref.abs().max()).all())
