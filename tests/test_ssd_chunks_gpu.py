"""The SSD with its chunks side by side (csrc/ssd_chunk.hpp), values and gradients, at the edges of its tiles: one step,
a step more or less than a chunk, a last chunk of a few rows, and every chunk and state size."""

import pytest
import torch

from oracle import ssd_oracle as S
from tests.test_ssd_gpu import DA_TERM_BAR_HALF, GRAD_ATOL_RMS, GRAD_MEAN_RMS, half_close, kernels_taken, ssd

pytestmark = pytest.mark.gpu

# (B, L, H, G, N), Q, options
CASES = [((1, 1, 1, 1, 64), 64, "z"), ((2, 65, 2, 1, 64), 64, "z init"), ((1, 192, 3, 1, 128), 64, "init final"),
         ((1, 127, 2, 2, 128), 128, "z"), ((2, 300, 4, 2, 64), 128, "z init final softplus"), ((1, 257, 3, 1, 128), 256, "z softplus"),
         ((2, 512, 2, 1, 128), 256, "z init final softplus clamp"), ((1, 700, 5, 1, 64), 256, "")]


def _inputs(shape, opts, dtype):
    b, l, h, g, n = shape
    gen = torch.Generator().manual_seed(l + n)
    r = lambda *s: torch.randn(*s, generator=gen)
    v = dict(x=r(b, l, h, 64).to(dtype), dt=r(b, l, h) * 0.5 if "softplus" in opts else torch.rand(b, l, h, generator=gen) * 0.3,
             A=-(torch.rand(h, generator=gen) + 0.2), B=(r(b, l, g, n) * 0.5).to(dtype), C=(r(b, l, g, n) * 0.5).to(dtype),
             D=r(h), z=r(b, l, h, 64).to(dtype) if "z" in opts else None, dt_bias=r(h) * 0.3 if "softplus" in opts else None,
             init=r(b, h, 64, n) if "init" in opts else None)
    return v, r(b, l, h, 64), r(b, h, 64, n) if "final" in opts else None


@pytest.mark.parametrize("shape,Q,opts", CASES, ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bfloat16", "float16"])
def test_values(shape, Q, opts, dtype):
    v, _, _ = _inputs(shape, opts, dtype)
    c = {k: None if t is None else t.cuda() for k, t in v.items()}
    limit = (0.1, 0.6) if "clamp" in opts else (0.0, float("inf"))
    for D in (v["D"], torch.randn(shape[2], 64, generator=torch.Generator().manual_seed(1))):
        call = lambda: ssd().ssd_combined(c["x"], c["dt"], c["A"], c["B"], c["C"], Q, D=D.cuda(), z=c["z"], dt_bias=c["dt_bias"],
                                          initial_states=c["init"], dt_softplus="softplus" in opts, dt_limit=limit,
                                          return_final_states=True)
        y, fin = call()
        assert kernels_taken(call) == 8
        dt = v["dt"].double() + (0.0 if v["dt_bias"] is None else v["dt_bias"].double())
        dt = (torch.nn.functional.softplus(dt) if "softplus" in opts else dt).clamp(*limit)
        wy, wf = S.ssd_sequential(v["x"], dt, v["A"], v["B"], v["C"], D=D, z=v["z"], initial_states=v["init"])
        half_close(y, wy, "y")
        half_close(fin, wf, "final states")


@pytest.mark.parametrize("shape,Q,opts", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_gradients(shape, Q, opts):
    b, l, h, g, n = shape
    v, dout, dfin = _inputs(shape, opts, torch.bfloat16)
    limit = (0.1, 0.6) if "clamp" in opts else (0.0, float("inf"))
    w = {k: None if t is None else t.double().requires_grad_() for k, t in v.items()}
    dt = w["dt"] if w["dt_bias"] is None else w["dt"] + w["dt_bias"]
    dt = (torch.nn.functional.softplus(dt) if "softplus" in opts else dt).clamp(*limit)
    A_steps = v["A"].double()[None, None].expand(b, l, h).clone().requires_grad_()     # dA term by term
    wy, wf = S.ssd_sequential(w["x"], dt, A_steps, w["B"], w["C"], D=w["D"], z=w["z"], initial_states=w["init"])
    ((wy * dout.double()).sum() + (0.0 if dfin is None else (wf * dfin.double()).sum())).backward()
    w["A"].grad = A_steps.grad.sum(dim=(0, 1))
    c = {k: None if t is None else t.cuda().requires_grad_() for k, t in v.items()}
    # the gradient is that of one stored number y whatever its rounding: dout enters in float32
    y, fin = ssd().ssd_combined(c["x"], c["dt"], c["A"], c["B"], c["C"], Q, D=c["D"], z=c["z"], dt_bias=c["dt_bias"],
                                initial_states=c["init"], dt_softplus="softplus" in opts, dt_limit=limit, return_final_states=True)
    assert type(y.grad_fn).__name__ != "SsdCombinedFnBackward"
    half_close(y, wy, "y")
    grads = torch.autograd.grad([y] if dfin is None else [y, fin], [t for t in c.values() if t is not None],
                                [dout.cuda().to(y.dtype)] if dfin is None else [dout.cuda().to(y.dtype), dfin.cuda()])
    for (k, t), got in zip([(k, t) for k, t in c.items() if t is not None], grads):
        want = w[k].grad
        assert got.dtype == t.dtype and got.shape == t.shape
        if k in ("A", "dt_bias"):         # sums over batch and time that cancel: against the magnitudes of their terms
            terms = (A_steps if k == "A" else w["dt"]).grad.abs().sum(dim=(0, 1))
            ratio = (got.cpu().double() - want).abs() / (terms + 1e-30)
            assert bool((ratio <= DA_TERM_BAR_HALF).all()), f"gradient of {k}: error / sum of magnitudes per head {ratio.tolist()}"
        else:
            half_close(got, want, f"gradient of {k}", atol_rms=GRAD_ATOL_RMS, mean_rms=GRAD_MEAN_RMS, rtol=3e-2)
