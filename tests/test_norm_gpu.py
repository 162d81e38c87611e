"""GPU parity of ``fused_layer_norm`` forward and backward against the CPU
oracle (autograd through it) and the upstream layer-norm vectors."""

import pytest
import torch

from oracle import ops_oracle as O
from tests import fixtures as fx

pytestmark = pytest.mark.gpu

FP32_TOL = dict(rtol=1e-5, atol=1e-5)
HALF_TOL = dict(rtol=2e-2, atol=2e-2)


def _ops():
    from ssm_amd import ops
    return ops


def cuda(t, grad=False):
    if t is None:
        return None
    t = t.clone().cuda()
    return t.requires_grad_(True) if grad else t


def run_pair(x, w, b, r, **kw):
    g = torch.Generator().manual_seed(17)
    go = torch.randn(x.shape, generator=g).to(x.dtype)
    out = []
    for where in ("gpu", "cpu"):
        if where == "gpu":
            xx, ww, bb, rr, gg = cuda(x, True), cuda(w, True), cuda(b, True), cuda(r, True), go.cuda()
            fn = _ops().fused_layer_norm
        else:
            xx, ww = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
            bb = b.clone().requires_grad_(True) if b is not None else None
            rr = r.clone().requires_grad_(True) if r is not None else None
            gg = go
            fn = O.fused_layer_norm
        y = fn(xx, ww, bb, residual=rr, **kw)
        y.backward(gg)
        out.append(dict(y=y.detach().cpu(), dx=xx.grad.cpu(), dw=ww.grad.cpu(),
                        db=bb.grad.cpu() if bb is not None else None,
                        dr=rr.grad.cpu() if rr is not None else None))
    return out


def check(pair, tol, ptol=None):
    got, want = pair
    for k in ("y", "dx", "dr"):
        if want[k] is not None:
            torch.testing.assert_close(got[k].float(), want[k].float(), **tol)
    for k in ("dw", "db"):
        if want[k] is not None:
            torch.testing.assert_close(got[k].float(), want[k].float(), **(ptol or tol))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,hidden", [(5001, 768), (5001, 704), (4097, 64), (2051, 1536), (1030, 4096), (517, 8192)])
@pytest.mark.parametrize("residual,bias,is_rms", [(False, False, True), (True, True, False), (True, False, True)])
def test_sums_over_rows_read_ahead(rows, hidden, dtype, residual, bias, is_rms):
    """More rows than owners, so that each walks several and asks for the next one ahead: the gradients against float64 of the same
    16-bit values.  Rows: one rounding of float32.  Weight and bias: sums of `rows` float32 terms of size about 1, whose rounding
    errors (2^-24 of a partial sum each) add up like a random walk, at most a few times 2^-24 x rows."""
    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, go = r(1, rows, hidden).to(dtype).requires_grad_(), r(1, rows, hidden).to(dtype)
    w, b = (r(hidden) + 1.0).requires_grad_(), r(hidden).requires_grad_() if bias else None
    res = r(1, rows, hidden).to(dtype).requires_grad_() if residual else None
    leaves = [t for t in (x, w, b, res) if t is not None]
    got = torch.autograd.grad(_ops().fused_layer_norm(x, w, b, residual=res, is_rms=is_rms, eps=1e-5), leaves, go)
    wide = [t.detach().double().requires_grad_() for t in leaves]
    v = wide[0] + wide[-1] if residual else wide[0]
    v = v if is_rms else v - v.mean(-1, keepdim=True)
    y = v * torch.rsqrt((v * v).mean(-1, keepdim=True) + 1e-5) * wide[1]
    want = torch.autograd.grad(y + wide[2] if bias else y, wide, go.double())
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for t, a, e in zip(leaves, got, want):
        tol = dict(rtol=eps, atol=1e-5) if t.dtype == dtype else dict(rtol=1e-5, atol=8 * 2.0 ** -24 * rows)
        torch.testing.assert_close(a.double(), e, **tol)


def test_upstream_layer_norm_prenorm():
    rec = fx.upstream("layer_norms", "layer_norm_prenorm")
    i = rec["inputs"]
    x, w, b, r = cuda(i["x"], True), cuda(i["w"], True), cuda(i["b"], True), cuda(i["residual"], True)
    y, res_out = _ops().fused_layer_norm_with_residual(x, w, b, residual=r, is_rms=False, eps=1e-6, prenorm=True,
                                                       residual_in_fp32=True)
    torch.testing.assert_close(y.cpu(), rec["outputs"]["y"], rtol=1e-4, atol=1e-5)
    torch.testing.assert_close(res_out.cpu(), rec["outputs"]["residual_out"], rtol=1e-5, atol=1e-6)
    y.sum().backward()
    for name, t in (("x", x), ("w", w), ("b", b), ("residual", r)):
        torch.testing.assert_close(t.grad.cpu(), rec["gradients"][name], rtol=1e-3, atol=2e-5)


def test_upstream_rms_norm():
    rec = fx.upstream("layer_norms", "rms_norm")
    i = rec["inputs"]
    x, w = cuda(i["x"], True), cuda(i["w"], True)
    y = _ops().fused_layer_norm(x, w, None, is_rms=True, eps=1e-6, prenorm=False, residual_in_fp32=False)
    torch.testing.assert_close(y.cpu(), rec["outputs"]["y"], rtol=1e-4, atol=1e-5)
    y.sum().backward()
    torch.testing.assert_close(x.grad.cpu(), rec["gradients"]["x"], rtol=1e-3, atol=2e-5)
    torch.testing.assert_close(w.grad.cpu(), rec["gradients"]["w"], rtol=1e-3, atol=2e-5)


@pytest.mark.parametrize("hidden", [1, 6, 64, 768, 770, 1024, 1536, 2048, 2500, 4096, 5120, 8192, 8200, 20000])
@pytest.mark.parametrize("is_rms", [False, True])
@pytest.mark.parametrize("prenorm", [True, False])
def test_fp32_matches_oracle(hidden, is_rms, prenorm):
    g = torch.Generator().manual_seed(hidden)
    x = torch.randn(2, 5, hidden, generator=g); r = torch.randn(2, 5, hidden, generator=g)
    w = torch.randn(hidden, generator=g); b = torch.randn(hidden, generator=g)
    check(run_pair(x, w, b, r, is_rms=is_rms, prenorm=prenorm, eps=1e-5), dict(rtol=1e-4, atol=1e-5),
          dict(rtol=1e-4, atol=1e-4))


def test_without_residual_and_bias():
    g = torch.Generator().manual_seed(3)
    x = torch.randn(3, 7, 96, generator=g); w = torch.randn(96, generator=g)
    check(run_pair(x, w, None, None, is_rms=True, eps=1e-5), dict(rtol=1e-4, atol=1e-5), dict(rtol=1e-4, atol=1e-4))
    check(run_pair(x, w, None, None, is_rms=False, eps=1e-5), dict(rtol=1e-4, atol=1e-5), dict(rtol=1e-4, atol=1e-4))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("is_rms", [False, True])
def test_half_input_fp32_residual(dtype, is_rms):
    g = torch.Generator().manual_seed(5)
    x = torch.randn(4, 64, 768, generator=g).to(dtype); r = torch.randn(4, 64, 768, generator=g)
    w = torch.randn(768, generator=g); b = torch.randn(768, generator=g)
    pair = run_pair(x, w, b, r, is_rms=is_rms, prenorm=True, eps=1e-5, residual_in_fp32=True)
    assert pair[0]["y"].dtype == dtype and pair[0]["dr"].dtype == torch.float32
    check(pair, HALF_TOL, dict(rtol=2e-2, atol=0.3))


def test_residual_out_matches_oracle_and_dtype_rules():
    g = torch.Generator().manual_seed(9)
    x = torch.randn(2, 9, 128, generator=g).to(torch.bfloat16); r = torch.randn(2, 9, 128, generator=g)
    w = torch.randn(128, generator=g)
    y, ro = _ops().fused_layer_norm_with_residual(x.cuda(), w.cuda(), None, residual=r.cuda(), is_rms=True)
    yr, ror = O.fused_layer_norm_with_residual(x, w, None, residual=r, is_rms=True)
    assert ro.dtype == torch.float32
    torch.testing.assert_close(ro.cpu(), ror, **FP32_TOL)
    torch.testing.assert_close(y.float().cpu(), yr.float(), **HALF_TOL)


def test_config4_layer_shape_bf16():
    """(16, 2048, 768) bf16 x with an fp32 residual stream, RMSNorm eps 1e-5: the shape of
    one fused add+norm in the 130M model.  Rows are independent, so a row slice is
    replayed on the oracle; dw/db are compared on that slice via linearity in rows."""
    g = torch.Generator().manual_seed(4)
    x = torch.randn(16, 2048, 768, generator=g).to(torch.bfloat16)
    r = torch.randn(16, 2048, 768, generator=g)
    w = torch.randn(768, generator=g)
    y, ro = _ops().fused_layer_norm_with_residual(x.cuda(), w.cuda(), None, residual=r.cuda(), is_rms=True)
    sl = slice(0, 2048, 97)
    yr, ror = O.fused_layer_norm_with_residual(x[:, sl], w, None, residual=r[:, sl], is_rms=True)
    torch.testing.assert_close(y[:, sl].float().cpu(), yr.float(), **HALF_TOL)
    torch.testing.assert_close(ro[:, sl].cpu(), ror, **FP32_TOL)


@pytest.mark.parametrize("is_rms", [True, False])
def test_postnorm_backward_with_a_residual_that_needs_no_gradient(is_rms):
    """bf16 x, float32 residual added after the norm, gradient asked for x and the weight only: the typed
    backward reads its stand-in for the unused residual from the residual itself (same type and extent)."""
    g = torch.Generator().manual_seed(8)
    x = torch.randn(3, 37, 768, generator=g).to(torch.bfloat16)
    r = torch.randn(3, 37, 768, generator=g)
    w = torch.randn(768, generator=g)
    gy = torch.randn(3, 37, 768, generator=g).to(torch.bfloat16)
    xg, wg = x.clone().cuda().requires_grad_(True), w.clone().cuda().requires_grad_(True)
    y = _ops().fused_layer_norm(xg, wg, None, residual=r.cuda(), is_rms=is_rms, prenorm=False)
    y.backward(gy.cuda())
    xr, wr = x.clone().float().requires_grad_(True), w.clone().requires_grad_(True)
    yr = O.fused_layer_norm(xr, wr, None, residual=r, is_rms=is_rms, prenorm=False)
    yr.backward(gy.float())
    torch.testing.assert_close(xg.grad.float().cpu(), xr.grad, rtol=2e-2, atol=2e-2)
    torch.testing.assert_close(wg.grad.cpu(), wr.grad, rtol=2e-2, atol=2e-2 * float(wr.grad.abs().max()))


@pytest.mark.parametrize("dtype,res_dtype,hidden", [
    (torch.bfloat16, torch.float32, 768), (torch.bfloat16, torch.bfloat16, 1028), (torch.float32, None, 100),
    (torch.bfloat16, None, 256), (torch.float16, torch.bfloat16, 64), (torch.float32, torch.float32, 8200), (torch.bfloat16, torch.float32, 37)])
@pytest.mark.parametrize("prenorm", [True, False])
def test_gradient_through_residual_out_is_added_in_the_backward_kernel(dtype, res_dtype, hidden, prenorm):
    """``residual_out = x (+ residual when prenorm)`` hands its gradient straight on: to ``dx``, and to the residual's
    when it was added before the norm -- for typed kernels (one type for residual and that gradient), mixed types,
    rows that are no multiple of four columns and rows beyond the register kernels."""
    g = torch.Generator().manual_seed(hidden)
    x, w = torch.randn(2, 5, hidden, generator=g).to(dtype), torch.randn(hidden, generator=g)
    r = None if res_dtype is None else torch.randn(2, 5, hidden, generator=g).to(res_dtype)
    gy, gr = torch.randn(2, 5, hidden, generator=g).to(dtype), torch.randn(2, 5, hidden, generator=g)
    xg, rg = x.cuda().requires_grad_(), None if r is None else r.cuda().requires_grad_()
    y, ro = _ops().fused_layer_norm_with_residual(xg, w.cuda(), None, residual=rg, is_rms=True, prenorm=prenorm)
    got = torch.autograd.grad([y, ro], [xg] + ([] if r is None else [rg]), [gy.cuda(), gr.cuda()])
    xd, rd = x.double().requires_grad_(), None if r is None else r.double().requires_grad_()
    s = xd if r is None or not prenorm else xd + rd
    out = s * torch.rsqrt((s * s).mean(-1, keepdim=True) + 1e-5) * w.double()
    if r is not None and not prenorm:
        out = out + rd
    want = torch.autograd.grad([out, s], [xd] + ([] if r is None else [rd]), [gy.double(), gr.double()])
    for a, b, t in zip(got, want, (x, r)):
        tol = 1e-5 if t.dtype == torch.float32 else 2e-2
        torch.testing.assert_close(a.double().cpu(), b, rtol=tol, atol=tol)


@pytest.mark.parametrize("dtype,res_dtype,hidden", [
    (torch.bfloat16, torch.float32, 768), (torch.float16, torch.float16, 2560), (torch.float32, torch.float32, 5120),
    (torch.bfloat16, torch.float32, 6148)])
def test_rows_of_a_large_call_are_those_of_its_halves(dtype, res_dtype, hidden):
    """Large calls read past the caches; a row does not depend on the others, so its results are the same to the bit."""
    rows = (3 << 20) // hidden                               # twice that: more elements than the caches are left, once: fewer
    g = torch.Generator(device="cuda").manual_seed(hidden)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, r, w = rand(2, rows, hidden).to(dtype), rand(2, rows, hidden).to(res_dtype), rand(hidden)
    go, gr = rand(2, rows, hidden).to(dtype), rand(2, rows, hidden).to(res_dtype)

    def run(part):
        leaves = [x[part].clone().requires_grad_(), r[part].clone().requires_grad_(), w.clone().requires_grad_()]
        y, out = _ops().fused_layer_norm_with_residual(leaves[0], leaves[2], None, residual=leaves[1], is_rms=True, eps=1e-5,
                                                       prenorm=True, residual_in_fp32=res_dtype == torch.float32)
        torch.autograd.backward([y, out], [go[part], gr[part]])
        return [y.detach(), out.detach()] + [t.grad for t in leaves]

    whole, halves = run(slice(None)), [run(slice(0, 1)), run(slice(1, 2))]
    for i in range(4):
        torch.testing.assert_close(whole[i], torch.cat([h[i] for h in halves]), rtol=0, atol=0)
    # the weight's gradient: sums of 2 `rows` products, any order off by at most 2 rows 2^-24 of the sum of their sizes
    v = x.double() + r.double()
    bound = 2 * rows * 2.0 ** -23 * (go.double() * v * (v * v).mean(-1, keepdim=True).add(1e-5).rsqrt()).abs().sum((0, 1))
    assert ((whole[4] - halves[0][4] - halves[1][4]).abs().double() <= bound).all()
