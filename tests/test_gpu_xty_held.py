"""Weight gradients with one operand held in registers (96 to 224 rows per expert on average, output rows on 128-byte lines):
expert loads on both sides of every slice boundary and of the 256 rows it holds, output sizes that are no whole number of
panels or steps, both output layouts, gathered rows, bias gradient, an output that is part of a larger one."""
import pytest
import torch

from scattermoe_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LOADS = [1, 63, 64, 65, 0, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 31, 600, 0, 90, 2]     # 148 on average


def _check(got, want, mass, n, dtype):
    """One rounding to the storage type, float32 sums of n products of total magnitude `mass` in any order."""
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    bound = unit * want.abs() + n * 2.0 ** -24 * mass + 2.0 ** -24
    assert bool(((got.double() - want).abs() <= bound).all())


def _inputs(K, N, dtype, k=2, loads=LOADS):
    g = torch.Generator(device=DEV).manual_seed(K + N)
    E, L = len(loads), sum(loads)
    assert L % k == 0 and 96 <= L // E <= 224 and E * -(-K // 256) * -(-N // 256) >= 256
    experts = torch.repeat_interleave(torch.arange(E, device=DEV), torch.tensor(loads, device=DEV))
    experts = experts[torch.randperm(L, generator=g, device=DEV)].view(L // k, k)
    _, idx, off = ops.route(experts, E)
    X = torch.randn(L // k, K, generator=g, device=DEV).to(dtype)
    DY = torch.randn(L, N, generator=g, device=DEV).to(dtype)
    return E, X, DY, idx, off, k


def _check_all(DW, Db, Xg, DY, off, dtype):
    lo = 0
    for e, hi in enumerate(off.tolist()):
        x, y = Xg[lo:hi].double(), DY[lo:hi].double()
        _check(DW[e], x.t() @ y, x.abs().t() @ y.abs(), hi - lo, dtype)
        if Db is not None:
            _check(Db[e], y.sum(0), y.abs().sum(0), hi - lo, dtype)
        lo = hi


# rows of dW: a whole number of 256-row panels, eight more, eight fewer; steps of 64 columns: one chunk of them or several
@pytest.mark.parametrize("K,N,layout", [(832, 1024, "nk"), (832, 1032, "nk"), (1024, 1016, "nk"), (1032, 832, "kn"),
                                        (1016, 6208, "kn")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_against_float64(K, N, layout, dtype):
    E, X, DY, idx, off, k = _inputs(K, N, dtype)
    like = torch.empty(E, K, N, dtype=dtype, device=DEV) if layout == "kn" else None
    Xg = ops.group(X, idx, fan_out=k)
    DW, Db = ops.group_bwd_W(DY, Xg, off, E, has_bias=True, like=like)
    DWg, Dbg = ops.group_bwd_W(DY, X, off, E, has_bias=True, like=like, gather=(idx, k))
    assert torch.equal(DW, DWg) and torch.equal(Db, Dbg)
    _check_all(DW, Db, Xg, DY, off, dtype)


def test_last_step_of_a_wider_output():
    """Columns that are no whole number of steps, in rows that start on 128-byte lines: nothing beside them is written."""
    E, X, DY, idx, off, k = _inputs(840, 1032, torch.bfloat16)
    Xg = ops.group(X, idx, fan_out=k)
    out = torch.full((E, 1032, 896), 7.0, dtype=torch.bfloat16, device=DEV)
    ops._xty_launch(E, out[:, :, :840].permute(0, 2, 1), None, DY, Xg, off)
    assert bool((out[:, :, 840:] == 7.0).all())
    _check_all(out[:, :, :840].permute(0, 2, 1), None, Xg, DY, off, torch.bfloat16)


@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_infinities_stay_with_their_expert(layout):
    """Rows of the next expert lie behind an expert's last one in both operands: they are not multiplied, not even by zero."""
    E, X, DY, idx, off, k = _inputs(832, 1024, torch.bfloat16)
    like = torch.empty(E, 832, 1024, dtype=torch.bfloat16, device=DEV) if layout == "kn" else None
    Xg = ops.group(X, idx, fan_out=k)
    want, want_b = ops.group_bwd_W(DY, Xg, off, E, has_bias=True, like=like)
    bad = 9                                                                # an expert of 192 rows
    lo, hi = off[bad - 1].item(), off[bad].item()
    Xg[lo:hi], DY[lo:hi] = float("inf"), float("nan")
    DW, Db = ops.group_bwd_W(DY, Xg, off, E, has_bias=True, like=like)
    keep = [e for e in range(E) if e != bad]
    assert torch.equal(DW[keep], want[keep]) and torch.equal(Db[keep], want_b[keep])
    assert bool(DW[bad].isnan().all())


# column steps of 64: one, two, three (fewer than there are stages), five
@pytest.mark.parametrize("width", [64, 128, 192, 320])
@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_few_steps_and_more_experts_than_a_wave_has_lanes(width, layout):
    """Experts of more than 256 rows in every group of 64."""
    K, N = (width, 512) if layout == "nk" else (512, width)
    E, X, DY, idx, off, k = _inputs(K, N, torch.bfloat16, loads=LOADS * 7)
    like = torch.empty(E, K, N, dtype=torch.bfloat16, device=DEV) if layout == "kn" else None
    DW, Db = ops.group_bwd_W(DY, X, off, E, has_bias=True, like=like, gather=(idx, k))
    _check_all(DW, Db, ops.group(X, idx, fan_out=k), DY, off, torch.bfloat16)


@pytest.mark.parametrize("which", ["DY", "X"])
@pytest.mark.parametrize("layout", ["nk", "kn"])
def test_rows_on_top_of_each_other(which, layout):
    """An expanded row as either operand: the same bits as of a copy."""
    E, X, DY, idx, off, k = _inputs(832, 1024, torch.bfloat16)
    t = {"DY": DY, "X": ops.group(X, idx, fan_out=k)}
    t[which] = t[which][:1].expand(DY.size(0), -1)
    like = torch.empty(E, 832, 1024, dtype=torch.bfloat16, device=DEV) if layout == "kn" else None
    DW, _ = ops.group_bwd_W(t["DY"], t["X"], off, E, like=like)
    want, _ = ops.group_bwd_W(t["DY"].contiguous(), t["X"].contiguous(), off, E, like=like)
    assert torch.equal(DW, want)
