"""The work whose speed counts: what a program built on ``ssm_amd.ops`` has the GPU do.

Nine kinds of work cover the public operators as blocks of a state-space model call them: the single-token steps of a
decoding loop, the scans of a prompt, and forward plus backward of a training step.  ``listed`` names one or two
sizes of each, from the smallest call to the largest; ``draw`` gives further sizes of the same kinds.
"""

from __future__ import annotations

import math

import torch

from ssm_amd import ops
from ssm_amd.configs import inverse_softplus_dt
from ssm_amd.ops import ssd

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
EPS = 1e-5


def listed():
    """One or two sizes of every kind of work."""
    return [
        # One token for a few sequences of a small block: nothing but latency (the reference's `decode_step_d512`).
        {"name": "state_step_d512", "op": "state_step", "batch": 4, "dim": 512, "nstate": 16, "dtype": "f32"},
        # One token of a wide Mamba-1 block with its convolution window, many sequences served together.
        {"name": "decode_step_d5120", "op": "decode_step", "batch": 64, "dim": 5120, "nstate": 16, "width": 4,
         "dtype": "bf16"},
        # One token of a Mamba-2 block of a 130M-parameter model.
        {"name": "mamba2_decode_130m", "op": "mamba2_decode", "batch": 16, "heads": 24, "nstate": 128, "width": 4,
         "dtype": "bf16"},
        # A single prompt through a small Mamba-1 block in float32 (the reference's `prefill_2k_d512`).
        {"name": "scan_prefill_2k_d512", "op": "scan", "batch": 1, "dim": 512, "seqlen": 2048, "nstate": 16,
         "dtype": "f32", "projection": "grouped", "train": False},
        # A batch of prompts through the Mamba-1 block of a 130M-parameter model, the state kept for decoding.
        {"name": "scan_prefill_130m", "op": "scan", "batch": 8, "dim": 1536, "seqlen": 2048, "nstate": 16,
         "dtype": "bf16", "projection": "grouped", "train": False},
        # A training step of the scan on sequences of no round length, in float32.
        {"name": "scan_train_ragged", "op": "scan", "batch": 3, "dim": 640, "seqlen": 1021, "nstate": 16,
         "dtype": "f32", "projection": "grouped", "train": True},
        # A training step of a Mamba-1 mixer: convolution, scan and all their gradients.
        {"name": "mamba1_mixer_train", "op": "mamba1_mixer", "batch": 8, "dim": 1536, "seqlen": 2048, "nstate": 16,
         "width": 4, "dtype": "bf16"},
        # A batch of long prompts through a wide Mamba-2 block.
        {"name": "ssd_prefill_4k_h80", "op": "ssd", "batch": 4, "seqlen": 4096, "heads": 80, "nstate": 128,
         "chunk": 256, "dtype": "bf16"},
        # One prompt that fills no whole number of chunks.
        {"name": "ssd_prefill_ragged", "op": "ssd", "batch": 1, "seqlen": 3001, "heads": 24, "nstate": 128,
         "chunk": 256, "dtype": "bf16"},
        # A training step of the Mamba-2 mixer of a 130M-parameter model: convolutions, SSD, gated norm, gradients.
        {"name": "mamba2_mixer_train", "op": "mamba2_mixer", "batch": 4, "seqlen": 2048, "heads": 24, "nstate": 128,
         "width": 4, "chunk": 256, "dtype": "bf16"},
        # A training step of the diagonal chunk scan as the reference's Mamba-2 module calls it (`chunk_scan_l2k_h16`).
        {"name": "chunk_scan_train", "op": "chunk_scan", "batch": 2, "seqlen": 2048, "heads": 16, "dtype": "f32",
         "form": "module", "train": True},
        # A training step of the residual-add RMSNorm between the blocks of a 130M-parameter model.
        {"name": "add_norm_train", "op": "add_norm", "batch": 16, "seqlen": 2048, "hidden": 768, "dtype": "bf16",
         "train": True},
    ]


def _between(rng, lo, hi, multiple=1):
    """A whole multiple from ``lo`` to ``hi``, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi // multiple, max(-(-lo // multiple), round(v / multiple))) * multiple


def _length(rng, lo, hi, most):
    """A sequence length of at most ``most``: any number half of the time, a multiple of 64 otherwise."""
    hi = max(lo, min(hi, most))
    return _between(rng, lo, hi, rng.choice([1, 64])) if hi >= 64 else _between(rng, lo, hi)


def draw(rng):
    """One more case: sizes over the range that the listed ones span."""
    op = rng.choice(["state_step", "decode_step", "mamba2_decode", "scan", "scan", "mamba1_mixer", "ssd",
                     "mamba2_mixer", "chunk_scan", "add_norm"])
    case = {"op": op, "dtype": rng.choice(["bf16", "bf16", "f32", "f16"])}
    if op in ("state_step", "decode_step"):
        case.update(batch=_between(rng, 1, 128), dim=_between(rng, 256, 5120, 16), nstate=16)
        if op == "decode_step":
            case.update(width=4)
    elif op == "mamba2_decode":
        case.update(batch=_between(rng, 1, 64), heads=_between(rng, 8, 80), nstate=rng.choice([64, 128]), width=4)
    elif op in ("scan", "mamba1_mixer"):
        batch, dim = _between(rng, 1, 8), _between(rng, 256, 2560, 16)
        case.update(batch=batch, dim=dim, nstate=16, seqlen=_length(rng, 128, 8192, 8 * 1536 * 2048 // (batch * dim)))
        if op == "scan":
            # B and C for all channels of a token, for every channel of its own, or the same at every token
            case.update(projection=rng.choice(["grouped", "grouped", "grouped", "per_channel", "constant"]),
                        train=rng.random() < 0.5)
            if case["projection"] == "per_channel":
                case["seqlen"] = max(64, case["seqlen"] // 4)
        else:
            case.update(width=4)
    elif op in ("ssd", "mamba2_mixer"):
        batch, heads = _between(rng, 1, 4), _between(rng, 8, 80)
        most = (4 * 4096 * 80 if op == "ssd" else 4 * 2048 * 24) // (batch * heads)
        case.update(batch=batch, heads=heads, seqlen=_length(rng, 256, 8192, most), nstate=rng.choice([64, 128]),
                    chunk=rng.choice([128, 256]), dtype=rng.choice(["bf16", "bf16", "f16"]) if op == "ssd" else "bf16")
        if op == "mamba2_mixer":
            case.update(width=4)
    elif op == "chunk_scan":
        batch, heads = _between(rng, 1, 4), _between(rng, 8, 80)
        case.update(batch=batch, heads=heads, seqlen=_length(rng, 256, 4096, 4 * 2048 * 40 // (batch * heads)),
                    dtype=rng.choice(["f32", "bf16"]), form=rng.choice(["module", "per_token"]),
                    train=rng.random() < 0.5)
    else:
        hidden = _between(rng, 256, 8192, 8)
        case.update(batch=_between(rng, 1, 16), hidden=hidden, train=rng.random() < 0.5)
        case.update(seqlen=_length(rng, 1, 4096, 16 * 2048 * 768 // (case["batch"] * hidden)))
    return case


def _maker(seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape, dtype=torch.float32, std=1.0):
        return torch.randn(*shape, generator=gen, device="cuda").mul_(std).to(dtype)

    def uniform(*shape, lo, hi):
        return torch.rand(*shape, generator=gen, device="cuda").mul_(hi - lo).add_(lo)

    def dt_bias(n):
        return inverse_softplus_dt(n, torch.Generator().manual_seed(seed)).cuda()

    return randn, uniform, dt_bias


def _mamba1_A(dim, nstate):
    return -torch.arange(1, nstate + 1, dtype=torch.float32, device="cuda").repeat(dim, 1).contiguous()


def prepare(case, seed):
    """Inputs, parameters and upstream gradients on the GPU."""
    c = dict(case)
    op, dt = c["op"], DTYPES[c["dtype"]]
    randn, uniform, dt_bias = _maker(seed)
    s = {"op": op}
    b = c["batch"]
    if op in ("state_step", "decode_step"):
        d, n = c["dim"], c["nstate"]
        s.update(state=randn(b, d, n), x=randn(b, d, dtype=dt), dt=randn(b, d, dtype=dt), A=_mamba1_A(d, n),
                 B=randn(b, 1, n, dtype=dt), C=randn(b, 1, n, dtype=dt), D=torch.ones(d, device="cuda"),
                 z=randn(b, d, dtype=dt), dt_bias=dt_bias(d))
        if op == "decode_step":
            s.update(window=randn(b, d, c["width"], dtype=dt), weight=uniform(d, c["width"], lo=-0.5, hi=0.5),
                     bias=randn(d, std=0.02))
    elif op == "mamba2_decode":
        h, p, n = c["heads"], 64, c["nstate"]
        di, conv = h * p, h * p + 2 * n
        s.update(row=randn(b, di + conv + h, dtype=dt), window=randn(b, conv, c["width"], dtype=dt),
                 state=randn(b, h, p, n), weight=uniform(conv, c["width"], lo=-0.5, hi=0.5), bias=randn(conv, std=0.02),
                 A=-uniform(h, lo=1.0, hi=16.0), D=torch.ones(h, device="cuda"), dt_bias=dt_bias(h))
    elif op in ("scan", "mamba1_mixer"):
        d, l, n = c["dim"], c["seqlen"], c["nstate"]
        kind = c.get("projection", "grouped")
        shape = {"grouped": (b, 1, n, l), "per_channel": (b, d, n, l), "constant": (d, n)}[kind]
        pdt = torch.float32 if kind == "constant" else dt
        s.update(u=randn(b, d, l, dtype=dt), delta=randn(b, d, l, dtype=dt), A=_mamba1_A(d, n), B=randn(*shape, dtype=pdt),
                 C=randn(*shape, dtype=pdt), D=torch.ones(d, device="cuda"), z=randn(b, d, l, dtype=dt),
                 dt_bias=dt_bias(d))
        names = ["u", "delta", "A", "B", "C", "D", "z", "dt_bias"]
        if op == "mamba1_mixer":
            s.update(weight=uniform(d, c["width"], lo=-0.5, hi=0.5), bias=randn(d, std=0.02))
            names += ["weight", "bias"]
        if op == "mamba1_mixer" or c["train"]:
            s.update(leaves=[s[k].requires_grad_() for k in names], grad=randn(b, d, l, dtype=dt))
    elif op in ("ssd", "mamba2_mixer"):
        l, h, p, n = c["seqlen"], c["heads"], 64, c["nstate"]
        s.update(dt=randn(b, l, h, dtype=dt), A=-uniform(h, lo=1.0, hi=16.0), D=torch.ones(h, device="cuda"),
                 dt_bias=dt_bias(h), chunk=c["chunk"])
        if op == "ssd":
            s.update(x=randn(b, l, h, p, dtype=dt), z=randn(b, l, h, p, dtype=dt), B=randn(b, l, 1, n, dtype=dt),
                     C=randn(b, l, 1, n, dtype=dt))
        else:
            s.update(x=randn(b, l, h * p, dtype=dt), bc=randn(b, l, 2 * n, dtype=dt), z=randn(b, l, h * p, dtype=dt),
                     weight_x=uniform(h * p, c["width"], lo=-0.5, hi=0.5), bias_x=randn(h * p, std=0.02),
                     weight_bc=uniform(2 * n, c["width"], lo=-0.5, hi=0.5), bias_bc=randn(2 * n, std=0.02),
                     norm=torch.ones(h * p, device="cuda"), grad=randn(b, l, h * p, dtype=dt))
            s["leaves"] = [s[k].requires_grad_() for k in ("x", "bc", "z", "dt", "A", "D", "dt_bias", "weight_x",
                                                           "bias_x", "weight_bc", "bias_bc", "norm")]
    elif op == "chunk_scan":
        l, h, p = c["seqlen"], c["heads"], 64
        module = c["form"] == "module"
        s.update(X=randn(b, l, h, p, dtype=dt),
                 dt=torch.nn.functional.softplus(randn(b, l, h) + dt_bias(h)), A=-uniform(h, p, lo=1.0, hi=16.0) if module
                 else -uniform(h, lo=1.0, hi=16.0), B=randn(h, p) if module else randn(b, l, h, p, dtype=dt),
                 C=randn(h, p) if module else randn(b, l, h, p, dtype=dt), D=randn(h, p) if module else randn(h),
                 z=None if module else randn(b, l, h, p, dtype=dt))
        if c["train"]:
            s["leaves"] = [s[k].requires_grad_() for k in ("X", "dt", "A", "B", "C", "D", "z") if s[k] is not None]
            s["grad"] = randn(b, l, h, p, dtype=dt)
    else:
        l, d = c["seqlen"], c["hidden"]
        s.update(x=randn(b, l, d, dtype=dt), residual=randn(b, l, d), weight=uniform(d, lo=0.5, hi=1.5))
        if c["train"]:
            s["leaves"] = [s[k].requires_grad_() for k in ("x", "residual", "weight")]
            s["grad"] = [randn(b, l, d, dtype=dt), randn(b, l, d)]
    return s


def _with_gradients(s, out):
    """The outputs and, in a training step, the gradients of every input and parameter."""
    out = list(out)
    if "leaves" not in s:
        return out
    grad = s["grad"] if isinstance(s["grad"], list) else [s["grad"]]
    return out + list(torch.autograd.grad(out, s["leaves"], grad))


def run(s):
    """One pass: a decoding step, a prefill, or forward and backward."""
    op = s["op"]
    if op == "state_step":
        y = ops.selective_state_step(s["state"], s["x"], s["dt"], s["A"], s["B"], s["C"], D=s["D"], z=s["z"],
                                     dt_bias=s["dt_bias"], softplus=True)
        return [y, s["state"]]
    if op == "decode_step":
        y = ops.decode_step(s["window"], s["state"], s["x"], s["dt"], s["A"], s["B"], s["C"], s["weight"], s["bias"],
                            D=s["D"], z=s["z"], dt_bias=s["dt_bias"], softplus=True)
        return [y, s["window"], s["state"]]
    if op == "mamba2_decode":
        y = ops.mamba2_decode_step(s["row"], s["window"], s["state"], s["weight"], s["bias"], s["A"], D=s["D"],
                                   dt_bias=s["dt_bias"])
        return [y, s["window"], s["state"]]
    if op in ("scan", "mamba1_mixer"):
        u = s["u"]
        if op == "mamba1_mixer":
            u = ops.dw_causal_conv(u, s["weight"], s["bias"], activation="silu")
        out = ops.selective_scan(u, s["delta"], s["A"], s["B"], s["C"], D=s["D"], z=s["z"], dt_bias=s["dt_bias"],
                                 softplus=True, return_last_state="leaves" not in s)
        return _with_gradients(s, out if isinstance(out, tuple) else [out])
    if op == "ssd":
        return list(ssd.ssd_combined(s["x"], s["dt"], s["A"], s["B"], s["C"], s["chunk"], D=s["D"], z=s["z"],
                                     dt_bias=s["dt_bias"], dt_softplus=True, return_final_states=True))
    if op == "mamba2_mixer":
        x = ops.dw_causal_conv_channels_last(s["x"], s["weight_x"], s["bias_x"], activation="silu")
        bc = ops.dw_causal_conv_channels_last(s["bc"], s["weight_bc"], s["bias_bc"], activation="silu")
        (b, l, h), n = s["dt"].shape, bc.shape[-1] // 2
        B, C = torch.split(bc, [n, n], dim=-1)
        y = ssd.ssd_combined(x.reshape(b, l, h, -1), s["dt"], s["A"], B.reshape(b, l, 1, n), C.reshape(b, l, 1, n),
                             s["chunk"], D=s["D"], z=s["z"].reshape(b, l, h, -1), dt_bias=s["dt_bias"],
                             dt_softplus=True)
        y = ops.fused_layer_norm(y.reshape(b, l, -1), s["norm"], None, is_rms=True, eps=EPS)
        return _with_gradients(s, [y])
    if op == "chunk_scan":
        return _with_gradients(s, [ops.ssd_chunk_scan(s["X"], s["dt"], s["A"], s["B"], s["C"], 128, D=s["D"], z=s["z"])])
    return _with_gradients(s, ops.fused_layer_norm_with_residual(s["x"], s["weight"], None, residual=s["residual"],
                                                                 is_rms=True, eps=EPS))


def work(case):
    """Bytes of every input read once and every output written once, and the arithmetic of one pass."""
    c = dict(case)
    op, e, b = c["op"], SIZE[c["dtype"]], c["batch"]
    if op in ("state_step", "decode_step"):
        d, n = c["dim"], c["nstate"]
        w = c.get("width", 0)
        return {"bytes": 8 * b * d * n + e * (4 * b * d + 2 * b * n + 2 * b * d * w) + 4 * d * (n + 2 + w + (w > 0)),
                "flops": b * d * (7 * n + 2 * w)}
    if op == "mamba2_decode":
        h, p, n = c["heads"], 64, c["nstate"]
        conv = h * p + 2 * n
        return {"bytes": 8 * b * h * p * n + e * b * (2 * h * p + conv + h + 2 * conv * c["width"])
                + 4 * (conv * (c["width"] + 1) + 3 * h), "flops": b * h * p * 6 * n + 2 * b * conv * c["width"]}
    if op in ("scan", "mamba1_mixer"):
        d, l, n = c["dim"], c["seqlen"], c["nstate"]
        kind, train = c.get("projection", "grouped"), op == "mamba1_mixer" or c["train"]
        proj = {"grouped": e * b * n * l, "per_channel": e * b * d * n * l, "constant": 4 * d * n}[kind]
        size = e * b * d * l
        moved, flops = 4 * size + 2 * proj + 4 * d * (n + 2), 7 * b * d * n * l
        if train:
            # u, delta, z and the upstream gradient again, three gradients and those of B and C
            moved, flops = moved + 7 * size + 4 * proj + 8 * d * (n + 2), 3 * flops
        else:
            moved += e * b * d * n
        if op == "mamba1_mixer":
            moved, flops = moved + 5 * size, flops + 6 * b * d * l * c["width"]
        return {"bytes": moved, "flops": flops}
    if op in ("ssd", "mamba2_mixer"):
        l, h, p, n, q = c["seqlen"], c["heads"], 64, c["nstate"], c["chunk"]
        size, proj = e * b * l * h * p, e * b * l * n
        # C.B of a chunk, its product with x, the states of the chunks and what they add
        flops = 2 * b * l * (q * n + h * (q * p + 2 * n * p))
        if op == "ssd":
            return {"bytes": 3 * size + 2 * proj + e * b * l * h + 4 * b * h * p * n + 12 * h, "flops": flops}
        # conv x: 2 + 3 tensors, SSD: 3 + 6, norm: 2 + 3; B and C through conv and SSD: 4 + 6 + 2 + 4; dt: 1 + 2
        return {"bytes": 19 * size + 16 * proj + 3 * e * b * l * h, "flops": 3 * flops}
    if op == "chunk_scan":
        l, h, p = c["seqlen"], c["heads"], 64
        size = b * l * h * p
        full = 1 if c["form"] == "module" else 4             # X alone, or X, B, C and z at every step
        moved = e * size * (full + 1) + 4 * b * l * h
        flops = 7 * size
        if c["train"]:
            moved, flops = moved + e * size * (2 * full + 1) + 8 * b * l * h, 3 * flops
        return {"bytes": moved, "flops": flops}
    l, d = c["seqlen"], c["hidden"]
    size = b * l * d
    moved, flops = size * (2 * e + 8) + 4 * d, 6 * size
    if c["train"]:
        # x and the residual again with both upstream gradients, and the gradients of x and the residual
        moved, flops = moved + size * (3 * e + 12) + 8 * d, 3 * flops
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """What another order of the same float32 sums, or one rounding to 16 bits more or less, changes."""
    train = case["op"] in ("mamba1_mixer", "mamba2_mixer") or case.get("train", False)
    if case["dtype"] == "f32":
        # gradients of parameters are sums over every token that largely cancel
        return {"rel": 1e-4 if train else 1e-5}
    if case["op"] == "mamba2_mixer":
        # the gradients of A and dt_bias are such sums, of products of rounded operands
        return {"rel": 3e-2, "max": 0.5}
    return {"rel": 1e-2}
