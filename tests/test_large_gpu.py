"""Tensors of more than 2**31 elements (the entry points promise 2**40): every kernel forms its addresses in
64 bits, or from a 64-bit base and a small 32-bit offset.  An address that wraps shows as garbage, not as a
rounding difference, so each operator is checked through a property that needs no oracle at this size: its rows
(channels, heads) are independent of each other, hence the last rows of the large call -- the ones whose
addresses lie beyond 2**32 bytes -- equal the same rows computed alone in a small call, and so do the first ones.
"""

import pytest
import torch

from tests.closeness import half_close

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _ops():
    from ssm_amd import ops
    return ops


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def test_selective_scan_forward_and_backward_beyond_2_31_elements():
    ops = _ops()
    batch, dim, length, nstate = 3, 3072, 262144 - 4096, 16
    assert batch * dim * length > 2 ** 31
    g = _gen(1)
    u, z = (torch.empty(batch, dim, length, device="cuda", dtype=BF).normal_(generator=g) for _ in range(2))
    delta = torch.empty(batch, dim, length, device="cuda", dtype=BF).normal_(generator=g)
    Bm, Cm = (torch.empty(batch, 1, nstate, length, device="cuda", dtype=BF).normal_(generator=g) for _ in range(2))
    A = -torch.arange(1, nstate + 1, device="cuda", dtype=torch.float32).repeat(dim, 1).contiguous()
    D = torch.ones(dim, device="cuda")
    bias = torch.full((dim,), -4.0, device="cuda")
    go = torch.empty(batch, dim, length, device="cuda", dtype=BF).normal_(generator=g)

    def run(b0, b1, d0, d1, grad):
        sl = lambda t: t[b0:b1, d0:d1].contiguous()
        lv = [sl(u), sl(delta), A[d0:d1].contiguous(), Bm[b0:b1].contiguous(), Cm[b0:b1].contiguous(),
              D[d0:d1].contiguous(), sl(z), bias[d0:d1].contiguous()]
        if grad:
            lv = [t.requires_grad_() for t in lv]
        y, last = ops.selective_scan(*lv[:5], D=lv[5], z=lv[6], dt_bias=lv[7], softplus=True, return_last_state=True)
        if not grad:
            return y, last, None
        y.backward(sl(go))
        return y.detach(), last.detach(), [t.grad for t in lv]

    y, last, grads = run(0, batch, 0, dim, True)
    torch.cuda.synchronize()
    for (b0, d0) in ((batch - 1, dim - 48), (0, 0), (1, 1536)):
        ys, lasts, gs = run(b0, b0 + 1, d0, d0 + 48, True)
        half_close(y[b0:b0 + 1, d0:d0 + 48].cpu(), ys.cpu(), what=f"y rows ({b0}, {d0}..)")
        half_close(last[b0:b0 + 1, d0:d0 + 48].cpu(), lasts.cpu(), what=f"last_state rows ({b0}, {d0}..)")
        for name, i in (("du", 0), ("ddelta", 1), ("dz", 6)):
            half_close(grads[i][b0:b0 + 1, d0:d0 + 48].cpu(), gs[i].cpu(), what=f"{name} rows ({b0}, {d0}..)",
                       atol_rms=4e-2, mean_rms=5e-3)


def test_causal_conv_beyond_2_31_elements():
    ops = _ops()
    batch, chans, length, width = 3, 3072, 262144 - 4096, 4
    g = _gen(2)
    x = torch.empty(batch, chans, length, device="cuda", dtype=BF).normal_(generator=g)
    go = torch.empty(batch, chans, length, device="cuda", dtype=BF).normal_(generator=g)
    w = torch.rand(chans, width, device="cuda", generator=g) - 0.5
    b = torch.randn(chans, device="cuda", generator=g) * 0.02
    y = ops._conv_forward(x, w, b, "silu")
    dx, _, _ = ops._conv_backward(go, x, w, b, "silu")
    for (b0, c0) in ((batch - 1, chans - 8), (0, 0)):
        xs, gs = x[b0:b0 + 1, c0:c0 + 8].contiguous(), go[b0:b0 + 1, c0:c0 + 8].contiguous()
        ws, bs = w[c0:c0 + 8].contiguous(), b[c0:c0 + 8].contiguous()
        half_close(y[b0:b0 + 1, c0:c0 + 8].cpu(), ops._conv_forward(xs, ws, bs, "silu").cpu(), what=f"y ({b0}, {c0}..)")
        half_close(dx[b0:b0 + 1, c0:c0 + 8].cpu(), ops._conv_backward(gs, xs, ws, bs, "silu")[0].cpu(), what=f"dx ({b0}, {c0}..)")
    # channels last: the same bytes read as (B, L', C') with C' = 2048 channels
    xl, gl = x.view(batch, -1, 2048), go.view(batch, -1, 2048)
    wl, bl = w[:2048].contiguous(), b[:2048].contiguous()
    yl = ops._conv_forward(xl, wl, bl, "silu", channels_last=True)
    dxl, _, _ = ops._conv_backward(gl, xl, wl, bl, "silu", channels_last=True)
    for (b0, c0) in ((batch - 1, 2040), (0, 0)):
        xs, gs = xl[b0:b0 + 1, :, c0:c0 + 8].contiguous(), gl[b0:b0 + 1, :, c0:c0 + 8].contiguous()
        ws, bs = wl[c0:c0 + 8].contiguous(), bl[c0:c0 + 8].contiguous()
        half_close(yl[b0:b0 + 1, :, c0:c0 + 8].cpu(), ops._conv_forward(xs, ws, bs, "silu", channels_last=True).cpu(),
                   what=f"channels last y ({b0}, {c0}..)")
        half_close(dxl[b0:b0 + 1, :, c0:c0 + 8].cpu(), ops._conv_backward(gs, xs, ws, bs, "silu", channels_last=True)[0].cpu(),
                   what=f"channels last dx ({b0}, {c0}..)")


def test_view_of_rows_beyond_2_31_elements():
    """The permuted view of (B, L, C) rows that the reference's blocks pass: the convolution reads it as it lies
    (forward and backward) and ``dense_copy`` turns it, at more than 2**31 elements."""
    ops = _ops()
    from ssm_amd.ops import _contract as K
    batch, length, chans, width = 3, 387072, 2048, 4
    assert batch * length * chans > 2 ** 31
    g = _gen(6)
    rows = torch.empty(batch, length, chans, device="cuda", dtype=BF).normal_(generator=g)
    w = torch.rand(chans, width, device="cuda", generator=g) - 0.5
    b = torch.randn(chans, device="cuda", generator=g) * 0.02
    x = rows.permute(0, 2, 1)
    assert ops._conv_rows_view(x, True, width) is not None
    y = ops._conv_forward(x, w, b, "silu")
    for (b0, c0) in ((batch - 1, chans - 8), (0, 0)):
        xs = x[b0:b0 + 1, c0:c0 + 8].contiguous()
        ws, bs = w[c0:c0 + 8].contiguous(), b[c0:c0 + 8].contiguous()
        assert torch.equal(y[b0:b0 + 1, c0:c0 + 8], ops._conv_forward(xs, ws, bs, "silu")), (b0, c0)
    go = y                                   # any (B, C, L) tensor of the type serves as the incoming gradient
    dx, _, _ = ops._conv_backward(go, x, w, b, "silu")
    assert dx.shape == x.shape and dx.stride() == (length * chans, 1, chans)
    for (b0, c0) in ((batch - 1, chans - 8), (0, 0)):
        xs, gs = x[b0:b0 + 1, c0:c0 + 8].contiguous(), go[b0:b0 + 1, c0:c0 + 8].contiguous()
        ws, bs = w[c0:c0 + 8].contiguous(), b[c0:c0 + 8].contiguous()
        assert torch.equal(dx[b0:b0 + 1, c0:c0 + 8], ops._conv_backward(gs, xs, ws, bs, "silu")[0]), (b0, c0)
    del dx, go
    dense = K.dense_copy(x)
    assert dense.is_contiguous()
    for (b0, c0) in ((batch - 1, chans - 8), (1, 1000), (0, 0)):
        assert torch.equal(dense[b0, c0:c0 + 8], x[b0, c0:c0 + 8]), (b0, c0)


def test_fused_norm_beyond_2_31_elements():
    ops = _ops()
    rows, hidden = 2_900_000, 768
    assert rows * hidden > 2 ** 31
    g = _gen(3)
    x = torch.empty(1, rows, hidden, device="cuda", dtype=BF).normal_(generator=g)
    res = torch.empty(1, rows, hidden, device="cuda", dtype=BF).normal_(generator=g)
    go = torch.empty(1, rows, hidden, device="cuda", dtype=BF).normal_(generator=g)
    w = torch.randn(hidden, device="cuda", generator=g)
    y, ro, mean, rstd = ops._norm_forward(x, w, None, res, True, 1e-5, True, False, want_residual_out=True, want_stats=True)
    dx, dres, _, _ = ops._norm_backward(go, x, w, res, mean, rstd, True, True, False, True)
    for r0 in (rows - 64, 0):
        xs, rs, gs = (t[:, r0:r0 + 64].contiguous() for t in (x, res, go))
        ys, ros, ms, ss = ops._norm_forward(xs, w, None, rs, True, 1e-5, True, False, want_residual_out=True, want_stats=True)
        half_close(y[:, r0:r0 + 64].cpu(), ys.cpu(), what=f"y rows {r0}..")
        half_close(ro[:, r0:r0 + 64].cpu(), ros.cpu(), what=f"residual_out rows {r0}..")
        dxs, drs, _, _ = ops._norm_backward(gs, xs, w, rs, ms, ss, True, True, False, True)
        half_close(dx[:, r0:r0 + 64].cpu(), dxs.cpu(), what=f"dx rows {r0}..")
        half_close(dres[:, r0:r0 + 64].cpu(), drs.cpu(), what=f"dresidual rows {r0}..")


def test_diagonal_chunk_scan_beyond_2_31_elements():
    ops = _ops()
    batch, seqlen, heads, proj = 2, 200_000, 96, 64
    assert batch * seqlen * heads * proj > 2 ** 31
    g = _gen(4)
    X, Bm, Cm, z = (torch.empty(batch, seqlen, heads, proj, device="cuda", dtype=BF).normal_(generator=g) for _ in range(4))
    dt = torch.rand(batch, seqlen, heads, device="cuda", generator=g) * 0.1
    A = -(torch.rand(heads, device="cuda", generator=g) + 0.5)
    D = torch.ones(heads, device="cuda")
    Y = ops.ssd_chunk_scan(X, dt, A, Bm, Cm, 256, D=D, z=z)
    for (b0, h0) in ((batch - 1, heads - 2), (0, 0)):
        sl = lambda t: t[b0:b0 + 1, :, h0:h0 + 2].contiguous()
        Ys = ops.ssd_chunk_scan(sl(X), sl(dt), A[h0:h0 + 2].contiguous(), sl(Bm), sl(Cm), 256, D=D[h0:h0 + 2].contiguous(), z=sl(z))
        half_close(Y[b0:b0 + 1, :, h0:h0 + 2].cpu(), Ys.cpu(), what=f"Y heads ({b0}, {h0}..)")


def test_ssd_combined_beyond_2_31_elements():
    from ssm_amd.ops import ssd
    batch, seqlen, heads, hdim, nstate, Q = 1, 262144 + 65536, 112, 64, 128, 256
    assert batch * seqlen * heads * hdim > 2 ** 31
    g = _gen(5)
    x, z = (torch.empty(batch, seqlen, heads, hdim, device="cuda", dtype=BF).normal_(generator=g) for _ in range(2))
    Bm, Cm = (torch.empty(batch, seqlen, 1, nstate, device="cuda", dtype=BF).normal_(generator=g) for _ in range(2))
    dt = torch.rand(batch, seqlen, heads, device="cuda", generator=g) * 0.1
    A = -(torch.rand(heads, device="cuda", generator=g) * 15 + 1)
    D = torch.ones(heads, device="cuda")
    y, final = ssd.ssd_combined(x, dt, A, Bm, Cm, Q, D=D, z=z, return_final_states=True)
    for h0 in (heads - 2, 0):
        sl = lambda t: t[:, :, h0:h0 + 2].contiguous()
        ys, fs = ssd.ssd_combined(sl(x), sl(dt), A[h0:h0 + 2].contiguous(), Bm, Cm, Q, D=D[h0:h0 + 2].contiguous(), z=sl(z),
                                  return_final_states=True)
        # the large call runs the five kernels (a batch row beyond the one-pass kernel's 32-bit offsets), the two heads
        # alone the one-pass kernel: two 16-bit paths that round at different places, compared over 42 M elements --
        # the bar on single elements is the tail of that difference (seen: 0.16 rms in one element), the mean stays
        # at the usual level; a wrapped address gives errors of the order of the values themselves everywhere
        half_close(y[:, :, h0:h0 + 2].cpu(), ys.cpu(), what=f"y heads {h0}..", atol_rms=0.3)
        half_close(final[:, h0:h0 + 2].cpu(), fs.cpu(), what=f"final states heads {h0}..", atol_rms=0.3)


@pytest.mark.parametrize("varying", [False, True])
def test_one_row_of_more_than_2_32_bytes(varying):
    """Two rows of float32 whose ends lie more than 2**32 bytes behind their starts, few enough for their chunks to run side by
    side.  The state forgets within tens of steps (it falls by e^-1 and e^-2 at each), so from 300 steps before 2**30 on the
    outputs are those of a call that begins 724 steps earlier, a whole number of chunks into the row, up to the rounding of
    sums of float32."""
    ops = _ops()
    dim, length, cut = 2, 2 ** 30 + 4 * 512 + 5, 2 ** 30 - 1024
    g = _gen(3)
    u = torch.empty(1, dim, length, device="cuda").normal_(generator=g)
    delta = torch.empty(1, dim, length, device="cuda").fill_(1.0)
    A = -torch.tensor([[1.0, 2.0]], device="cuda").repeat(dim, 1)
    if varying:
        B, C = (torch.empty(1, 1, 2, length, device="cuda").normal_(generator=g) for _ in range(2))
    else:
        B, C = (torch.randn(dim, 2, generator=g, device="cuda") for _ in range(2))
    y, last = ops.selective_scan(u, delta, A, B, C, return_last_state=True)
    part = lambda t: t[..., cut:].contiguous()
    ys, lasts = ops.selective_scan(part(u), part(delta), A, part(B) if varying else B, part(C) if varying else C,
                                   return_last_state=True)
    torch.testing.assert_close(y[..., cut + 724:], ys[..., 724:], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(last, lasts, rtol=1e-5, atol=1e-5)
