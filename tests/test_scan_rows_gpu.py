"""Scan rows that are no whole aligned runs, and calls of few rows whose chunks run side by side: forward and backward
against float64 autograd through the oracle, at the edges of runs (8 and 16 steps), chunks (512 steps), the walks of
1024 steps and the eight chunks a workgroup takes at once; and the end of a tensor, which no read may pass."""

import pytest
import torch

from oracle import ops_oracle as O
from tests.test_scan_fwd_gpu import make_inputs

pytestmark = pytest.mark.gpu
NAMES = ("u", "delta", "A", "B", "C", "D", "z", "dt_bias")


def _close(a, b, half, what, scale_tol):
    a, b = a.detach().double().cpu(), b.detach().double()
    scale = float(b.abs().max()) + 1e-30
    tol = dict(rtol=2e-2, atol=4e-3 * scale) if half else dict(rtol=1e-3, atol=scale_tol * scale)
    torch.testing.assert_close(a, b, **tol, msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("kind", ["grouped", "own", "dn"])
@pytest.mark.parametrize("length,dim,dtype,use_z", [
    (511, 16, torch.float32, True), (513, 48, torch.bfloat16, True), (519, 16, torch.float16, False),
    (1021, 96, torch.bfloat16, True), (1025, 16, torch.float32, True), (1543, 24, torch.float32, True),
    (4097, 16, torch.float32, False), (4608, 16, torch.bfloat16, True)])
def test_rows_of_any_length(kind, length, dim, dtype, use_z):
    from ssm_amd import ops
    if kind == "own" and length > 2048:
        length = length % 2048 + 520
    kw = dict(groups=dim) if kind == "own" else dict(groups=1) if kind == "grouped" else dict(bkind="dn", ckind="dn")
    inp = make_inputs(length, 2, dim, length, 16, dtype=dtype, bc_dtype=torch.float32 if kind == "dn" else dtype, use_z=use_z, **kw)
    g = torch.Generator().manual_seed(1)
    go, gl = torch.randn(2, dim, length, generator=g).to(dtype), torch.randn(2, dim, 16, generator=g).to(dtype)
    got = {k: (None if v is None else v.cuda().requires_grad_(True)) for k, v in inp.items()}
    want = {k: (None if v is None else v.double().requires_grad_(True)) for k, v in inp.items()}
    y, h = ops.selective_scan(*(got[k] for k in NAMES[:5]), D=got["D"], z=got["z"], dt_bias=got["dt_bias"], softplus=True,
                              return_last_state=True)
    yr, hr = O.selective_scan(*(want[k] for k in NAMES[:5]), D=want["D"], z=want["z"], dt_bias=want["dt_bias"], softplus=True,
                              return_last_state=True, acc=torch.float64)
    half = dtype != torch.float32
    _close(y, yr, half, "y", 1e-5)
    _close(h, hr, half, "last state", 1e-5)
    with torch.no_grad():
        y0 = ops.selective_scan(*(got[k] for k in NAMES[:5]), D=got["D"], z=got["z"], dt_bias=got["dt_bias"], softplus=True)
    assert torch.equal(y0, y)
    torch.autograd.backward([y, h], [go.cuda(), gl.cuda()])
    torch.autograd.backward([yr, hr], [go.double(), gl.double()])
    for k in NAMES:
        if want[k] is not None:
            _close(got[k].grad, want[k].grad, half and got[k].dtype == dtype, f"grad {k}", 1e-4)


def test_many_rows_of_odd_length_walk_their_chunks_in_turn():
    """Enough rows that no chunk runs beside another (workgroups of 8 channels forward, of 16 backward): the same
    numbers as the first rows computed alone, which take the other kernels."""
    from ssm_amd import ops
    inp = make_inputs(7, 4, 1040, 521, 16, dtype=torch.float32, groups=1)
    go = torch.randn(4, 1040, 521, generator=torch.Generator().manual_seed(2)).cuda()

    def run(batch):
        t = {k: (v[:batch] if k in ("u", "delta", "z", "B", "C") else v).cuda().requires_grad_(True) for k, v in inp.items()}
        y = ops.selective_scan(*(t[k] for k in NAMES[:5]), D=t["D"], z=t["z"], dt_bias=t["dt_bias"], softplus=True)
        y.backward(go[:batch].contiguous())
        return [y] + [t[k].grad for k in ("u", "delta", "z", "B", "C")]
    for a, b, what in zip(run(4), run(1), ("y", "u", "delta", "z", "B", "C")):
        scale = float(b.detach().abs().max())
        torch.testing.assert_close(a[:1], b, rtol=1e-4, atol=2e-5 * scale, msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("batch,dim,length,nstate,dtype", [
    (3, 344, 1543, 16, torch.float32), (2, 648, 4112, 16, torch.float32), (2, 1016, 1040, 5, torch.float32),
    (2, 800, 2064, 16, torch.bfloat16), (2, 496, 1537, 9, torch.float16), (3, 488, 2063, 16, torch.bfloat16)])
def test_rows_shared_by_two_waves(batch, dim, length, nstate, dtype):
    """Rows so few that two waves take each, with half of the states: the numbers of the first batch row alone, whose chunks
    run side by side in another kernel."""
    from ssm_amd import ops
    inp = make_inputs(length, batch, dim, length, nstate, dtype=dtype, bc_dtype=dtype, groups=1)
    g = torch.Generator().manual_seed(2)
    go, gl = torch.randn(batch, dim, length, generator=g).to(dtype).cuda(), torch.randn(batch, dim, nstate, generator=g).to(dtype).cuda()

    def run(rows):
        t = {k: (v[:rows] if k in ("u", "delta", "z", "B", "C") else v).cuda().requires_grad_(True) for k, v in inp.items()}
        y, h = ops.selective_scan(*(t[k] for k in NAMES[:5]), D=t["D"], z=t["z"], dt_bias=t["dt_bias"], softplus=True,
                                  return_last_state=True)
        torch.autograd.backward([y, h], [go[:rows].contiguous(), gl[:rows].contiguous()])
        return [y, h] + [t[k].grad for k in ("u", "delta", "z", "B", "C")]
    for a, b, what in zip(run(batch), run(1), ("y", "last state", "u", "delta", "z", "B", "C")):
        a, b = a.detach()[:1].float(), b.detach().float()
        # both sum in float32; a 16-bit result may be rounded to either neighbour
        tol = dict(rtol=1e-4, atol=2e-5) if dtype == torch.float32 else dict(rtol=2.0 ** -7, atol=1e-4)
        torch.testing.assert_close(a, b, rtol=tol["rtol"], atol=tol["atol"] * float(b.abs().max()), msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_what_lies_past_a_row_never_enters_it(dtype):
    """The row after next holds infinities: steps past the end of a row are read with it and must count for nothing."""
    from ssm_amd import ops
    inp = make_inputs(3, 2, 16, 515, 16, dtype=dtype, groups=1)
    t = {k: (None if v is None else v.cuda()) for k, v in inp.items()}
    call = lambda: ops.selective_scan(*(t[k] for k in NAMES[:5]), D=t["D"], z=t["z"], dt_bias=t["dt_bias"], softplus=True,
                                      return_last_state=True)
    y, h = call()
    for k in ("u", "delta", "z", "B", "C"):
        t[k][1] = float("inf")
    y2, h2 = call()
    assert torch.equal(y2[0], y[0]) and torch.equal(h2[0], h[0])


@pytest.mark.parametrize("length,dtype", [(1, torch.float32), (15, torch.bfloat16), (64, torch.float32), (195, torch.bfloat16),
                                          (256, torch.float16)])
def test_short_rows_with_projections_per_channel(length, dtype):
    test_rows_of_any_length("own", length, 16, dtype, True)


@pytest.mark.parametrize("batch,dim,length,nstate,dtype,bc_dtype,groups", [
    (3, 688, 1031, 16, torch.float32, torch.float32, (1, 1)),      # 2064 rows: nine to a workgroup, the last of a batch has fewer
    (8, 400, 1544, 15, torch.bfloat16, torch.bfloat16, (1, 1)),    # thirteen: a second turn of one row; odd number of states
    (4, 1616, 521, 16, torch.float16, torch.float16, (1, 1)),      # 26: three turns, a last chunk of nine steps
    (6, 576, 1027, 9, torch.bfloat16, torch.float32, (4, 6)),      # runs of 48 channels share B and C
    (9, 2720, 264, 16, torch.float32, torch.float32, (2, 1)),      # 24480 rows: one round of 96
    (5, 304, 256, 16, torch.bfloat16, torch.bfloat16, (1, 1)), (5, 304, 251, 11, torch.float32, torch.float32, (1, 4)),
    (2, 24, 4, 16, torch.float16, torch.float16, (1, 1)), (2, 12, 7, 16, torch.bfloat16, torch.float32, (1, 1))])
def test_any_number_of_channels_to_a_workgroup(batch, dim, length, nstate, dtype, bc_dtype, groups):
    """The channels at a batch row's and a group's edges against float64, and the state after each chunk through the
    gradients' entry; what lies in other rows (infinities beyond the compared ones) stays there."""
    from ssm_amd import ops
    inp = make_inputs(length, batch, dim, length, nstate, dtype=dtype, bc_dtype=bc_dtype, groups=1)
    g = torch.Generator().manual_seed(1)
    inp["B"], inp["C"] = (torch.randn(batch, n, nstate, length, generator=g).to(bc_dtype) for n in groups)
    pick = sorted({0, 1, 11, 12 % dim, dim // 2, dim - 2, dim - 1})
    for k in ("u", "delta"):
        inp[k][:, [d for d in range(dim) if d not in pick and d % 5 == 0], -1] = float("inf")
    t = {k: v.cuda() for k, v in inp.items()}
    y, h = ops.selective_scan(*(t[k] for k in NAMES[:5]), D=t["D"], z=t["z"], dt_bias=t["dt_bias"], softplus=True,
                              return_last_state=True)
    part = {k: v[:, pick] for k, v in inp.items() if k in ("u", "delta", "z")}
    part.update({k: inp[k][pick] for k in ("A", "D", "dt_bias")})
    for k, n in zip("BC", groups):
        part[k] = inp[k][:, [d // (dim // n) for d in pick]]
    yr, hr = O.selective_scan(*(part[k].double() for k in NAMES[:5]), D=part["D"].double(), z=part["z"].double(),
                              dt_bias=part["dt_bias"].double(), softplus=True, return_last_state=True, acc=torch.float64)
    half = dtype != torch.float32
    # one rounding of the float32 result to 16 bits (or of sums over the states to float32)
    tol = dict(rtol=2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -10, atol=1e-4) if half else dict(rtol=1e-5, atol=1e-5)
    for a, b, what in ((y[:, pick], yr, "y"), (h[:, pick], hr, "last state")):
        scale = float(b.abs().max())
        torch.testing.assert_close(a.double().cpu(), b, rtol=tol["rtol"], atol=tol["atol"] * scale, msg=lambda m: f"{what}: {m}")


@pytest.mark.parametrize("batch,dim,length,nstate,dtype,bc_dtype,groups,rows", [
    (8, 3072, 265, 16, torch.float32, torch.float32, (1, 1), 96), (8, 3072, 277, 15, torch.bfloat16, torch.float32, (1, 1), 96),
    (16, 1440, 64, 16, torch.float16, torch.float16, (1, 1), 90), (9, 2720, 264, 16, torch.float32, torch.float32, (2, 1), 49)])
def test_the_largest_workgroups(batch, dim, length, nstate, dtype, bc_dtype, groups, rows):
    """Workgroups of as many channels as fit (the most rows to a wave and LDS), and of a size that leaves one over."""
    from ssm_amd import _lib
    assert _lib.load_test_hooks().ssm_scan_fwd_rows_per_workgroup(batch, dim, length, *groups) == rows
    test_any_number_of_channels_to_a_workgroup(batch, dim, length, nstate, dtype, bc_dtype, groups)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("length,nstate", [(403, 1), (403, 15), (403, 16), (1031, 3), (200, 9), (200, 16)])
def test_an_infinite_step_stays_where_it_is(length, nstate, dtype):
    """An infinite u reaches the outputs from its own step on, as an infinity where nothing cancels it; the steps ahead of it,
    those in the same lane's run among them, are what they were."""
    from ssm_amd import ops
    inp = make_inputs(length, 2, 24 if length < 1031 else 520, length, nstate, dtype=dtype, groups=1)
    t = {k: v.cuda() for k, v in inp.items()}
    for k in ("B", "C", "D"):
        t[k] = t[k].abs() + 0.1
    call = lambda: ops.selective_scan(*(t[k] for k in NAMES[:5]), D=t["D"], dt_bias=t["dt_bias"], softplus=True)
    clean = call()
    rows = torch.arange(t["u"].shape[1], device="cuda")
    at = 100 + rows % 24                                    # every place in a run of 16
    t["u"][:, rows, at] = float("inf")
    y = call()
    ahead = (torch.arange(length, device="cuda") < at[:, None]).expand_as(y)
    assert torch.equal(y[ahead], clean[ahead])
    assert (y[:, rows, at] == float("inf")).all()
