"""The native host path of repeated calls (``ssm_amd/csrc/host/host.cpp``): the second call of a form, which goes
through the remembered argument struct, gives the bits of the first, which goes through every check -- values,
gradients and in-place updates -- and calls that the struct does not describe still go the long way."""

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _rand(seed, *shape, dtype=torch.float32, grad=False):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(dtype).cuda().requires_grad_(grad)


def _scan(dtype, grad, kind="grouped", L=640):
    b, d, n = 2, 32, 16
    shape = {"grouped": (b, 1, n, L), "own": (b, d, n, L), "dn": (d, n)}[kind]
    pt = torch.float32 if kind == "dn" else dtype
    t = [_rand(1, b, d, L, dtype=dtype, grad=grad), _rand(2, b, d, L, dtype=dtype, grad=grad),
         (-torch.rand(d, n).cuda() - 0.5).requires_grad_(grad), _rand(4, *shape, dtype=pt, grad=grad),
         _rand(5, *shape, dtype=pt, grad=grad), _rand(6, d, grad=grad), _rand(7, b, d, L, dtype=dtype, grad=grad),
         _rand(8, d, grad=grad)]
    return t, lambda o, u, dl, A, B, C, D, z, bias: o.selective_scan(u, dl, A, B, C, D=D, z=z, dt_bias=bias, softplus=True,
                                                                     return_last_state=True)


def _conv(dtype, grad, last):
    x = _rand(1, 2, 96, 24, dtype=dtype, grad=grad) if last else _rand(1, 2, 24, 96, dtype=dtype, grad=grad)
    t = [x, _rand(2, 24, 1, 4, dtype=dtype, grad=grad), _rand(3, 24, grad=grad)]
    f = "dw_causal_conv_channels_last" if last else "dw_causal_conv"
    return t, lambda o, x, w, b: getattr(o, f)(x, w, b, activation="silu")


def _norm(dtype, grad, res, prenorm=True, with_res_out=True, hidden=192):
    t = [_rand(1, 2, 9, hidden, dtype=dtype, grad=grad), _rand(2, hidden, grad=grad), _rand(3, hidden, grad=grad)]
    if res is not None:
        t.append(_rand(4, 2, 9, hidden, dtype=res, grad=grad))

    def call(o, x, w, b, r=None):
        f = o.fused_layer_norm_with_residual if with_res_out else o.fused_layer_norm
        return f(x, w, b, residual=r, is_rms=False, prenorm=prenorm, residual_in_fp32=res != BF)
    return t, call


def _chunk(dtype, grad, module):
    b, L, h, p = 2, 150, 3, 64
    small = (h, p) if module else (b, L, h, p)
    t = [_rand(1, b, L, h, p, dtype=dtype, grad=grad), torch.rand(b, L, h).cuda().requires_grad_(grad),
         (-torch.rand(*((h, p) if module else (h,))).cuda() - 0.5).requires_grad_(grad),
         _rand(4, *small, dtype=torch.float32 if module else dtype, grad=grad),
         _rand(5, *small, dtype=torch.float32 if module else dtype, grad=grad), _rand(6, h, grad=grad)]
    return t, lambda o, X, dt, A, B, C, D: o.ssd_chunk_scan(X, dt, A, B, C, 64, D=D)


CASES = [("scan", _scan, (torch.float32,)), ("scan", _scan, (BF,)), ("scan", _scan, (BF, "own")), ("scan", _scan, (torch.float16, "dn")),
         ("conv", _conv, (BF, True)), ("conv", _conv, (torch.float32, False)),
         ("norm", _norm, (BF, torch.float32)), ("norm", _norm, (BF, BF)), ("norm", _norm, (torch.float32, None)),
         ("norm", _norm, (BF, torch.float32, False)), ("norm", _norm, (BF, None, True, False)),
         ("chunk", _chunk, (torch.float32, True)), ("chunk", _chunk, (BF, False))]


@pytest.mark.parametrize("name,make,args", CASES, ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else None)
def test_a_repeated_call_gives_the_bits_of_the_first(name, make, args):
    from ssm_amd import ops
    forms = {"scan": ops._SCAN_FORMS, "conv": ops._CONV_FORMS, "norm": ops._NORM_FORMS, "chunk": ops._CHUNK_FORMS}[name]
    forms.clear()
    for grad in (False, True):
        t, call = make(args[0], grad, *args[1:])
        got = []
        for again in range(2):
            out = call(ops, *t)
            out = list(out) if isinstance(out, tuple) else [out]
            if grad:
                out += torch.autograd.grad(out, t, [_rand(20 + i, *o.shape, dtype=o.dtype) for i, o in enumerate(out)])
                assert [g.dtype for g in out[-len(t):]] == [x.dtype for x in t]
            got.append([o.detach().clone() for o in out])
            assert len(forms) == 1                     # one form, with gradients or without
            if not grad or again:
                continue
            forms.clear()                              # the first call with gradients takes the long way as well
            out = call(ops, *t)
            out = list(out) if isinstance(out, tuple) else [out]
            out += torch.autograd.grad(out, t, [_rand(20 + i, *o.shape, dtype=o.dtype) for i, o in enumerate(out)])
            got[0] = [o.detach().clone() for o in out]
        for a, b in zip(*got):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, BF])
def test_decoding_steps_repeat_their_bits(dtype):
    from ssm_amd import ops
    b, d, n, k, h = 3, 64, 16, 4, 2
    for f in (ops._DECODE_FORMS, ops._MAMBA2_FORMS, ops._WINDOW_FORMS):
        f.clear()
    win, st = _rand(1, b, d, k, dtype=dtype), _rand(2, b, d, n)
    x, dt, z = (_rand(i, b, d, dtype=dtype) for i in (3, 4, 5))
    B, C = (_rand(i, b, 1, n, dtype=dtype) for i in (6, 7))
    A, w = -torch.rand(d, n).cuda() - 0.5, _rand(8, d, k)
    row, win2, st2 = _rand(9, b, 2 * h * 64 + 2 * n + h, dtype=dtype), _rand(10, b, h * 64 + 2 * n, k, dtype=dtype), _rand(11, b, h, 64, n)
    A2, w2 = -torch.rand(h).cuda(), _rand(12, h * 64 + 2 * n, k)
    wide = _rand(13, b, 2 * d, dtype=dtype)[:, :d]
    got = []
    for _ in range(2):
        a, s, a2, s2, c = win.clone(), st.clone(), win2.clone(), st2.clone(), win.clone()
        got.append([ops.decode_step(a, s, x, dt, A, B, C, w, None, z=z), a, s, ops.mamba2_decode_step(row, a2, s2, w2, None, A2),
                    a2, s2, ops.conv_window_step(c, wide, w), c])
    for p, q in zip(*got):
        assert torch.equal(p, q)
    assert len(ops._DECODE_FORMS) == len(ops._MAMBA2_FORMS) == len(ops._WINDOW_FORMS) == 1
    with pytest.raises(ValueError):                    # a form never seen, and inconsistent
        ops.decode_step(win, st, x, dt, A, B, C, w[:, :3].contiguous(), None, z=z)


def test_one_pass_ssd_repeats_its_bits_on_views_of_one_projection():
    from ssm_amd.ops import ssd
    ssd._FUSED_FORMS.clear()
    b, L, h, n = 1, 128, 2, 64
    x, z, dt = _rand(1, b, L, h, 64, dtype=BF), _rand(2, b, L, h, 64, dtype=BF), _rand(3, b, L, h, dtype=BF)
    B, C = (t.reshape(b, L, 1, n) for t in torch.split(_rand(4, b, L, 2 * n, dtype=BF), [n, n], dim=-1))
    A, D = -torch.rand(h).cuda() - 1, _rand(5, h)
    got = [ssd.ssd_combined(x, dt, A, B, C, 64, D=D, z=z, dt_softplus=True, return_final_states=True) for _ in range(2)]
    assert len(ssd._FUSED_FORMS) == 1
    for p, q in zip(*got):
        assert torch.equal(p, q)
