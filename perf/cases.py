"""The calls whose time this framework is judged by: what a program built on it
has it do, through the public entry points, from one decode step of one
sequence to training layers over thousands of steps.

A case is a dict of plain values whose ``kind`` names the entry point:

==============  ==================================================================
update          ``selective_state_update``: one decode step of the SSM state
scan            ``selective_scan_fn`` without autograd: prefill of one layer
scan_train      the scan forward and backward (``SelectiveScanFn`` without the
                gate, ``selective_scan_fn`` with it): every gradient
conv_train      ``causal_conv1d_fn`` forward and backward
block_train     ``Block`` forward and backward: every gradient of the layer
block_prefill   ``Block`` without autograd, filling the decode caches
block_step      ``Block.step``: one token per sequence, caches advancing
lm_step         ``CausalLM.step``: one token through a whole model, to its logits
==============  ==================================================================

Inputs follow the reference's initialisation and activation scales: A = -(1 ..
N), D = 1, step sizes of softplus^-1 of a log-uniform step in [1e-3, 1e-1].
"""
import math

import torch
import torch.nn.functional as F

from ssm_mamba_amd.causal_conv1d import causal_conv1d_fn
from ssm_mamba_amd.causal_lm import Block, CausalLM, CausalLMConfig
from ssm_mamba_amd.ops import SelectiveScanFn, selective_scan_fn, selective_state_update

DEV = "cuda"
DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp32": 4}


def listed():
    return [
        # one sequence decoded by a program that owns its own loop: the smallest call
        dict(name="update-1", kind="update", batch=1, dim=2048, nstate=16, dtype="bf16", gate=True),
        # a serving batch of 64 on a wide model: the decode benchmark's shape
        dict(name="update-64", kind="update", batch=64, dim=5120, nstate=16, dtype="bf16",
             gate=True),
        # a short float32 prompt, as the reference's float32 operators are used
        dict(name="scan-short", kind="scan", batch=2, dim=1536, seqlen=512, nstate=16,
             dtype="fp32", gate=True, lengths="none"),
        # the scan of a 370M-class training step: the headline benchmark
        dict(name="scan-train", kind="scan_train", batch=8, dim=2048, seqlen=2048, nstate=16,
             dtype="bf16", gate=True, lengths="none"),
        # one long document in float32
        dict(name="scan-train-long", kind="scan_train", batch=1, dim=2560, seqlen=16384, nstate=16,
             dtype="fp32", gate=True, lengths="none"),
        # a left-padded batch of odd length and width through the reference's own operator
        dict(name="scan-train-ragged", kind="scan_train", batch=3, dim=1000, seqlen=1531, nstate=16,
             dtype="fp32", gate=False, lengths="left"),
        # a model with a larger state
        dict(name="scan-train-n64", kind="scan_train", batch=4, dim=1024, seqlen=1000, nstate=64,
             dtype="bf16", gate=True, lengths="none"),
        # the short convolution of a training step
        dict(name="conv-train", kind="conv_train", batch=4, dim=2048, seqlen=2048, width=4,
             dtype="bf16", bias=True),
        # one layer of a training step
        dict(name="block-train", kind="block_train", batch=4, seqlen=2048, model_dim=1024,
             nstate=16, dtype="bf16", lengths="none"),
        # one layer of a prefill over a left-padded batch, caches kept for decoding
        dict(name="block-prefill", kind="block_prefill", batch=4, seqlen=2048, model_dim=1024,
             nstate=16, dtype="bf16", lengths="left"),
        # one layer of a decode step for 32 sequences served together
        dict(name="block-step-32", kind="block_step", batch=32, model_dim=1024, nstate=16,
             dtype="bf16"),
        # one token for 4 sequences through a whole model
        dict(name="lm-step", kind="lm_step", batch=4, model_dim=1024, layers=24, vocab=50280,
             nstate=16, dtype="bf16"),
    ]


# ---------------------------------------------------------------- drawn cases


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["update", "scan", "scan_train", "scan_train", "scan_train", "conv_train",
                       "block_train", "block_prefill", "block_step", "lm_step"])
    dtype = rng.choice(["bf16", "bf16", "fp32"])
    gate = rng.random() < 0.7
    pad = rng.choice(["none", "none", "left", "right"])
    nstate = rng.choice([16, 16, 16, 8, 32, 64])
    if kind == "update":
        return dict(kind=kind, batch=_log(rng, 1, 64), dim=_log(rng, 96, 5120), nstate=nstate,
                    dtype=dtype, gate=gate)
    if kind in ("scan", "scan_train"):
        batch, dim = _log(rng, 1, 8), _log(rng, 64, 2560)
        most = min(8192, (1 << 24) // (batch * dim * max(1, nstate // 16)))
        seqlen = _log(rng, 40, max(most, 64))
        if rng.random() < 0.6:  # most programs pad to a multiple of 8
            seqlen = (seqlen + 7) // 8 * 8
        return dict(kind=kind, batch=batch, dim=dim, seqlen=seqlen, nstate=nstate, dtype=dtype,
                    gate=gate, lengths=pad)
    if kind == "conv_train":
        batch, dim = _log(rng, 1, 8), _log(rng, 64, 2560)
        seqlen = _log(rng, 40, min(8192, (1 << 25) // (batch * dim)))
        if rng.random() < 0.6:
            seqlen = (seqlen + 7) // 8 * 8
        return dict(kind=kind, batch=batch, dim=dim, seqlen=seqlen, width=rng.choice([2, 3, 4, 4]),
                    dtype=dtype, bias=rng.random() < 0.5)
    model_dim = 8 * _log(rng, 8, 128)
    if kind in ("block_train", "block_prefill"):
        batch = _log(rng, 1, 8)
        seqlen = _log(rng, 40, min(4096, (1 << 22) // (batch * model_dim)))
        if rng.random() < 0.6:
            seqlen = (seqlen + 7) // 8 * 8
        return dict(kind=kind, batch=batch, seqlen=seqlen, model_dim=model_dim, nstate=16,
                    dtype=dtype, lengths=rng.choice(["none", "left"]))
    if kind == "block_step":
        return dict(kind=kind, batch=_log(rng, 1, 64), model_dim=model_dim, nstate=16, dtype=dtype)
    return dict(kind=kind, batch=_log(rng, 1, 16), model_dim=model_dim,
                layers=rng.randrange(2, 13), vocab=rng.choice([32000, 50280]), nstate=16,
                dtype=dtype)


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dtype)


def _step_bias(g, dim):
    lo, hi = math.log(1e-3), math.log(1e-1)
    dt = torch.exp(torch.rand(dim, generator=g, device=DEV) * (hi - lo) + lo).clamp(min=1e-4)
    return dt + torch.log(-torch.expm1(-dt))


def _lengths(g, case):
    if case["lengths"] == "none":
        return None
    n = case["seqlen"]
    r = torch.rand(case["batch"], generator=g, device=DEV) * 0.75 + 0.25
    r[0] = 1.0
    return (r * n).long().clamp(1, n)


def _ssm_inputs(g, case, io):
    b, d, n = case["batch"], case["dim"], case["nstate"]
    tail = (case["seqlen"],) if "seqlen" in case else ()
    return dict(
        u=_randn(g, (b, d) + tail, io), delta=_randn(g, (b, d) + tail, io, 0.5),
        A=-torch.arange(1, n + 1, device=DEV, dtype=torch.float32).repeat(d, 1),
        B=_randn(g, (b, n) + tail, io), C=_randn(g, (b, n) + tail, io),
        D=1.0 + _randn(g, (d,), torch.float32, 0.1),
        z=_randn(g, (b, d) + tail, io) if case["gate"] else None,
        bias=_step_bias(g, d))


def _seeded_module(make, seed, io):
    with torch.random.fork_rng(devices=[torch.device(DEV, torch.cuda.current_device())]):
        torch.manual_seed(seed)
        m = make().to(DEV)
        with torch.no_grad():  # the norms start at zero: give them trained-looking scales
            for name, p in m.named_parameters():
                if name.endswith("norm.weight"):
                    p.normal_(0.0, 0.1)
                if name.endswith("D"):
                    p.normal_(1.0, 0.1)
    return m.to(io)


def _fill_caches(g, blocks, batch, io):
    for blk in blocks:
        blk.ssm.allocate_cache(batch)
        blk.ssm._conv_context.copy_(_randn(g, blk.ssm._conv_context.shape, io, 0.5))
        blk.ssm._ssm_hiddens.copy_(_randn(g, blk.ssm._ssm_hiddens.shape, torch.float32, 0.1))


def prepare(case, seed):
    kind, io, g = case["kind"], DT[case["dtype"]], _gen(seed)
    s = dict(case=case)
    if kind == "update":
        s.update(_ssm_inputs(g, case, io))
        s["state"] = _randn(g, (case["batch"], case["dim"], case["nstate"]), torch.float32, 0.1)
    elif kind in ("scan", "scan_train"):
        s.update(_ssm_inputs(g, case, io))
        s["length"] = _lengths(g, case)
        if kind == "scan_train":
            s["dout"] = _randn(g, s["u"].shape, io)
            for k in ("u", "delta", "A", "B", "C", "D", "z", "bias"):
                if s[k] is not None:
                    s[k].requires_grad_(True)
    elif kind == "conv_train":
        b, d, n, w = case["batch"], case["dim"], case["seqlen"], case["width"]
        s["x"] = _randn(g, (b, d, n), io).requires_grad_(True)
        s["w"] = _randn(g, (d, 1, w), io, w ** -0.5).requires_grad_(True)
        s["b"] = _randn(g, (d,), io, 0.2).requires_grad_(True) if case["bias"] else None
        s["dout"] = _randn(g, (b, d, n), io)
    elif kind in ("block_train", "block_prefill", "block_step"):
        # the layer of the model's default configuration; a training step's
        # dropout draws other numbers in each pass, so it is off here
        m = _seeded_module(lambda: Block(model_dim=case["model_dim"], state_dim=case["nstate"],
                                         dropout_rate=0.0, device=DEV), seed, io)
        s["block"] = m.train() if kind == "block_train" else m.eval()
        if kind == "block_step":
            _fill_caches(g, [m], case["batch"], io)
            s["x"] = _randn(g, (case["batch"], case["model_dim"]), io)
        else:
            shape = (case["batch"], case["seqlen"], case["model_dim"])
            s["x"] = _randn(g, shape, io)
            s["length"] = _lengths(g, case)
            if kind == "block_train":
                s["x"].requires_grad_(True)
                s["dout"] = _randn(g, shape, io)
            else:
                m.ssm.allocate_cache(case["batch"])
    else:
        cfg = CausalLMConfig(vocab_size=case["vocab"], model_dim=case["model_dim"],
                             state_dim=case["nstate"], num_layers=case["layers"], device=DEV)
        m = _seeded_module(lambda: CausalLM(cfg), seed, io).eval()
        _fill_caches(g, m.layers, case["batch"], io)
        s["model"] = m
        s["ids"] = torch.randint(3, case["vocab"], (case["batch"],), generator=g, device=DEV)
    return s


# ---------------------------------------------------------------- one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "update":
        out = selective_state_update(s["state"], s["u"], s["delta"], s["A"], s["B"], s["C"], s["D"],
                                     z=s["z"], dt_bias=s["bias"])
        return {"out": out, "state": s["state"]}
    if kind == "scan":
        with torch.no_grad():
            out, last = selective_scan_fn(
                s["u"], s["delta"], s["A"], s["B"], s["C"], s["D"], z=s["z"], delta_bias=s["bias"],
                return_last_state=True, length=s["length"], padding_side=_side(case))
        return {"out": out, "last": last}
    if kind == "scan_train":
        if case["gate"]:
            out, last = selective_scan_fn(
                s["u"], s["delta"], s["A"], s["B"], s["C"], s["D"], z=s["z"], delta_bias=s["bias"],
                return_last_state=True, length=s["length"], padding_side=_side(case))
        else:
            out, last = SelectiveScanFn.apply(s["u"], s["A"], s["B"], s["C"], s["D"], s["delta"],
                                              s["bias"], None, s["length"], _side(case))
        names = [k for k in ("u", "delta", "A", "B", "C", "D", "z", "bias") if s[k] is not None]
        grads = torch.autograd.grad(out, [s[k] for k in names], s["dout"])
        return {"out": out, "last": last, **{"d" + k: v for k, v in zip(names, grads)}}
    if kind == "conv_train":
        out = causal_conv1d_fn(s["x"], s["w"], s["b"])
        names = [k for k in ("x", "w", "b") if s[k] is not None]
        grads = torch.autograd.grad(out, [s[k] for k in names], s["dout"])
        return {"out": out, **{"d" + k: v for k, v in zip(names, grads)}}
    if kind == "block_train":
        blk = s["block"]
        out, last = blk(s["x"], lengths=s["length"])
        names, params = zip(*blk.named_parameters())
        grads = torch.autograd.grad(out, [s["x"], *params], s["dout"])
        return {"out": out, "last": last, "dx": grads[0], **dict(zip(names, grads[1:]))}
    if kind == "block_prefill":
        blk = s["block"]
        with torch.no_grad():
            out, last = blk(s["x"], lengths=s["length"], use_cache=True)
        return {"out": out, "last": last, "window": blk.ssm._conv_context,
                "state": blk.ssm._ssm_hiddens}
    if kind == "block_step":
        blk = s["block"]
        with torch.no_grad():
            out = blk.step(s["x"])
        return {"out": out, "window": blk.ssm._conv_context, "state": blk.ssm._ssm_hiddens}
    m = s["model"]
    with torch.no_grad():
        logits = m.step(s["ids"])
    return {"logits": logits, "windows": [b.ssm._conv_context for b in m.layers],
            "states": [b.ssm._ssm_hiddens for b in m.layers]}


def _side(case):
    return "right" if case["lengths"] == "right" else "left"


# ---------------------------------------------------------------- what a pass cannot do without


def _block_sizes(case):
    """(inner, rank, weights of the projections, all parameters) of a layer."""
    k = case["model_dim"]
    inner, rank, n = 2 * k, math.ceil(k / 16), case["nstate"]
    proj = 2 * inner * k + inner * (rank + 2 * n) + inner * rank + inner * k
    return inner, rank, proj, proj + k + inner * (4 + 1 + n + 1)


def work(case):
    kind, e = case["kind"], SIZE[case["dtype"]]
    n, b = case.get("nstate", 0), case["batch"]
    gate = 1 if case.get("gate") else 0
    if kind == "update":
        d = case["dim"]
        return {"bytes": 8 * b * d * n + e * b * (d * (3 + gate) + 2 * n) + 4 * d * (n + 2),
                "flops": b * d * (7 * n + 10)}
    if kind in ("scan", "scan_train"):
        d, t = case["dim"], case["seqlen"]
        el, small = b * d * t, 4 * d * (n + 2)
        fwd = e * (el * (3 + gate) + 2 * b * n * t) + small + 4 * b * d * n
        if kind == "scan":
            return {"bytes": fwd, "flops": el * (7 * n + 10)}
        bwd = e * (el * (5 + 2 * gate) + 4 * b * n * t) + 2 * small
        return {"bytes": fwd + bwd, "flops": el * (27 * n + 30)}
    if kind == "conv_train":
        d, t, w = case["dim"], case["seqlen"], case["width"]
        return {"bytes": e * (5 * b * d * t + 2 * d * (w + 1)), "flops": b * d * t * (8 * w + 12)}
    if kind == "lm_step":
        inner, _, proj, params = _block_sizes(case)
        head = case["vocab"] * case["model_dim"]
        state = b * inner * (8 * n + 2 * 3 * e)
        return {"bytes": case["layers"] * (e * params + state) + e * (head + b * case["vocab"]),
                "flops": 2 * b * (case["layers"] * proj + head)}
    inner, _, proj, params = _block_sizes(case)
    k = case["model_dim"]
    if kind == "block_step":
        return {"bytes": e * (params + 2 * b * k) + b * inner * (8 * n + 2 * 3 * e),
                "flops": 2 * b * proj + b * inner * 7 * n}
    tok = b * case["seqlen"]
    scan = tok * inner * 7 * n
    if kind == "block_prefill":
        return {"bytes": e * (params + 2 * tok * k) + b * inner * (8 * n + 3 * e),
                "flops": 2 * tok * proj + scan}
    return {"bytes": e * (2 * params + 4 * tok * k) + 4 * b * inner * n,
            "flops": 6 * tok * proj + 4 * scan}


def tolerance(case):
    # four times the largest distance from the same pass in 64 bits, over these
    # cases and their ranges, rounded up: one rounding of the results to bf16
    # (2e-3) or a float32 sum (1e-6) for a single operator; the roundings of
    # a layer's intermediate tensors on top for a layer (prefill 4.3e-3,
    # gradients 8.4e-3 in bf16 and 2.2e-6 in float32); those of all layers
    # for a model's logits (8e-3)
    bf16 = case["dtype"] == "bf16"
    return {
        "update": {"rel": 1e-2 if bf16 else 1e-5},
        "scan": {"rel": 1e-2 if bf16 else 1e-5},
        "scan_train": {"rel": 1e-2 if bf16 else 1e-5},
        "conv_train": {"rel": 1e-2 if bf16 else 1e-5},
        "block_train": {"rel": 3e-2 if bf16 else 1e-5},
        "block_prefill": {"rel": 2e-2 if bf16 else 1e-5},
        "block_step": {"rel": 1e-2 if bf16 else 1e-5},
        "lm_step": {"rel": 3e-2 if bf16 else 1e-5},
    }[case["kind"]]


# ---------------------------------------------------------------- the same in 64 bits


def _f64(t):
    return None if t is None else t.detach().double()


def _scan64(u, delta, A, B, C, D, z, bias, length, side):
    """Gated scan and last state, differentiable; the scan's outputs at padded
    positions carry no gradient."""
    b, d, n = u.shape
    dt = F.softplus(delta + bias[None, :, None])
    pos = torch.arange(n, device=u.device)
    if length is None:
        valid = None
    else:
        lo = n - length if side == "left" else torch.zeros_like(length)
        hi = torch.full_like(length, n) if side == "left" else length
        valid = ((pos >= lo[:, None]) & (pos < hi[:, None]))[:, None]
        dt = dt * valid
    h = u.new_zeros(b, d, A.shape[1])
    ys = []
    for t0 in range(0, n, 64):
        sl = slice(t0, t0 + 64)
        a = torch.exp(dt[:, :, sl].permute(2, 0, 1)[..., None] * A)
        x = (dt * u)[:, :, sl].permute(2, 0, 1)[..., None] * B[:, :, sl].permute(2, 0, 1)[:, :, None]
        hs = []
        for at, xt in zip(a.unbind(0), x.unbind(0)):
            h = torch.addcmul(xt, at, h)
            hs.append(h)
        ys.append(torch.einsum("tbdn,bnt->bdt", torch.stack(hs), C[:, :, sl]))
    y = torch.cat(ys, dim=2) + D[None, :, None] * u
    if valid is not None:
        y = torch.where(valid, y, y.detach())
    return (y if z is None else y * F.silu(z)), h


def _norm64(x, w, eps=1e-6):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * (1.0 + w)


def _block64(p, x, nstate, length):
    """(out, last state, pre-conv inputs) of one layer, token-major x."""
    h = _norm64(x, p["norm.weight"])
    xs, z = (h @ p["ssm.input_proj.weight"].t()).transpose(1, 2).chunk(2, dim=1)
    k = p["ssm.conv.weight"].shape[-1]
    xc = F.silu(F.conv1d(F.pad(xs, (k - 1, 0)), p["ssm.conv.weight"], groups=xs.shape[1]))
    prm = (xc.transpose(1, 2) @ p["ssm.ssm_param_proj.weight"].t()).transpose(1, 2)
    r = prm.shape[1] - 2 * nstate
    delta = (prm[:, :r].transpose(1, 2) @ p["ssm.delta_proj.weight"].t()).transpose(1, 2)
    y, last = _scan64(xc, delta, -torch.exp(p["ssm.log_A"]), prm[:, r:r + nstate],
                      prm[:, r + nstate:], p["ssm.D"], z, p["ssm.delta_proj.bias"], length, "left")
    return x + y.transpose(1, 2) @ p["ssm.out_proj.weight"].t(), last, xs


def _step64(p, x, window, state, nstate):
    """(out, window, state) of one token through one layer."""
    h = _norm64(x, p["norm.weight"])
    xs, z = (h @ p["ssm.input_proj.weight"].t()).chunk(2, dim=1)
    win = torch.cat([window, xs[..., None]], dim=-1)
    xc = F.silu((win * p["ssm.conv.weight"][:, 0]).sum(-1))
    prm = xc @ p["ssm.ssm_param_proj.weight"].t()
    r = prm.shape[1] - 2 * nstate
    dt = F.softplus(prm[:, :r] @ p["ssm.delta_proj.weight"].t() + p["ssm.delta_proj.bias"])
    B, C = prm[:, r:r + nstate], prm[:, r + nstate:]
    state = torch.exp(dt[..., None] * -torch.exp(p["ssm.log_A"])) * state \
        + (dt * xc)[..., None] * B[:, None]
    y = ((state * C[:, None]).sum(-1) + p["ssm.D"] * xc) * F.silu(z)
    return x + y @ p["ssm.out_proj.weight"].t(), win[..., 1:], state


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "update":
        v = {k: _f64(s[k]) for k in ("state", "u", "delta", "A", "B", "C", "D", "z", "bias")}
        dt = F.softplus(v["delta"] + v["bias"])
        state = torch.exp(dt[..., None] * v["A"]) * v["state"] \
            + (dt * v["u"])[..., None] * v["B"][:, None]
        out = (state * v["C"][:, None]).sum(-1) + v["D"] * v["u"]
        return {"out": out if v["z"] is None else out * F.silu(v["z"]), "state": state}
    if kind in ("scan", "scan_train"):
        v = {k: _f64(s[k]) for k in ("u", "delta", "A", "B", "C", "D", "z", "bias")}
        names = [k for k in v if v[k] is not None]
        if kind == "scan_train":
            for k in names:
                v[k].requires_grad_(True)
        out, last = _scan64(v["u"], v["delta"], v["A"], v["B"], v["C"], v["D"], v["z"], v["bias"],
                            s["length"], _side(case))
        res = {"out": out, "last": last}
        if kind == "scan_train":
            grads = torch.autograd.grad(out, [v[k] for k in names], _f64(s["dout"]))
            res.update({"d" + k: t for k, t in zip(names, grads)})
        return res
    if kind == "conv_train":
        v = {k: _f64(s[k]).requires_grad_(True) for k in ("x", "w", "b") if s[k] is not None}
        out = F.silu(F.conv1d(F.pad(v["x"], (case["width"] - 1, 0)), v["w"], v.get("b"),
                              groups=case["dim"]))
        grads = torch.autograd.grad(out, list(v.values()), _f64(s["dout"]))
        return {"out": out, **{"d" + k: t for k, t in zip(v, grads)}}
    if kind == "lm_step":
        m = s["model"]
        x = _f64(m.embedding.weight)[s["ids"]]
        windows, states = [], []
        for b in m.layers:
            p = {k: _f64(t) for k, t in b.named_parameters()}
            x, win, st = _step64(p, x, _f64(b.ssm._conv_context), _f64(b.ssm._ssm_hiddens),
                                 case["nstate"])
            windows.append(win)
            states.append(st)
        logits = _norm64(x, _f64(m.norm.weight)) @ _f64(m.lm_head.weight).t()
        return {"logits": logits, "windows": windows, "states": states}
    blk = s["block"]
    p = {k: _f64(t) for k, t in blk.named_parameters()}
    if kind == "block_step":
        out, win, st = _step64(p, _f64(s["x"]), _f64(blk.ssm._conv_context),
                               _f64(blk.ssm._ssm_hiddens), case["nstate"])
        return {"out": out, "window": win, "state": st}
    x = _f64(s["x"])
    if kind == "block_prefill":
        with torch.no_grad():
            out, last, xs = _block64(p, x, case["nstate"], s["length"])
        n, k = case["seqlen"], 4
        end = s["length"] if s["length"] is not None else torch.full((case["batch"],), n, device=DEV)
        at = end[:, None] - (k - 1) + torch.arange(k - 1, device=DEV)  # inputs ending at length - 1
        win = xs.gather(2, at.clamp(min=0)[:, None].expand(-1, xs.shape[1], -1)) * (at >= 0)[:, None]
        return {"out": out, "last": last, "window": win, "state": last}
    x.requires_grad_(True)
    for t in p.values():
        t.requires_grad_(True)
    out, last, _ = _block64(p, x, case["nstate"], s["length"])
    grads = torch.autograd.grad(out, [x, *p.values()], _f64(s["dout"]))
    return {"out": out, "last": last, "dx": grads[0], **dict(zip(p, grads[1:]))}
