"""Performance cases of the MoE block: what a program that uses it runs.

Kinds of work, each through the public binding (``tmt_moe``):

  forward  one forward of the block (bf16 or MXFP4 expert weights, with or
           without the LayerNorm in front): decode steps of 1 to 64 tokens,
           prompts, evaluation batches;
  train    one forward and backward (TMT's recurrent block calls exactly this
           pair per layer and step), aux and z loss on;
  norm     the standalone LayerNorm, forward and backward (TMT's MLA block);
  adamw    one multi-tensor AdamW step over a block's parameters.

The sizes are the ones of ``synthetic.CONFIGS``, of the benchmark's h = 0 legs
(the reference's profile shape and TMT's default width) and of the width
tests. Inputs follow ``synthetic.py``: activations N(0, 1), weights
N(0, 1/sqrt(fan_in)), made on the GPU from the seed alone.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "test-model-thing-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import tmt_moe  # noqa: E402

# -zipf * ln(e + 1) is the logit bias of expert e; 1.1 * 2.78 gives E = 16,
# top-4 a heaviest expert of about four times the mean load.
C3_ZIPF = 1.1 * 2.78

_FORMATS = {"bf16": tmt_moe.WEIGHTS_BF16, "mxfp4": tmt_moe.WEIGHTS_MXFP4,
            "mxfp4_mx": tmt_moe.WEIGHTS_MXFP4_MX, "mxfp4_planes": tmt_moe.WEIGHTS_MXFP4_MX_PLANES}


def _block(kind, T, d, E, K, h, weights="bf16", ln=False, zipf=0.0):
    return {"kind": kind, "T": T, "d": d, "E": E, "K": K, "h": h, "weights": weights, "ln": ln, "zipf": zipf}


def listed():
    big = dict(d=1024, E=16, K=4, h=4096)
    return [
        # Sampling one stream from the large model: the smallest call there is.
        dict(_block("forward", 1, **big), name="decode_1"),
        # A serving step over 64 streams, the largest decode batch.
        dict(_block("forward", 64, **big), name="decode_64"),
        # A serving step on quantised weights (they are what makes a decode
        # step cheaper), the exact format, LayerNorm outside.
        dict(_block("forward", 8, 1024, 32, 4, 4096, weights="mxfp4"), name="mxfp4_decode_8"),
        # A prompt of ragged length, or a small evaluation batch, forward only,
        # with the LayerNorm in front as the model has it.
        dict(_block("forward", 777, ln=True, **big), name="prefill_777"),
        # A training step's layer at TMT's default width (batch 8 x 128
        # tokens), reference experts, LayerNorm in front: launch-bound.
        dict(_block("train", 1024, 256, 4, 2, 0, ln=True), name="train_default_width"),
        # The shape the reference profiles its MoE layer at.
        dict(_block("train", 2048, 1280, 8, 2, 0), name="train_profile_shape"),
        # A mid-sized up/down model.
        dict(_block("train", 16384, 512, 8, 2, 2048), name="train_medium"),
        # Widths that are no multiple of 64 (any `dim=` is allowed), an odd
        # token count, top-3 of 12, LayerNorm in front, skewed routing.
        dict(_block("train", 5003, 1000, 12, 3, 2730, ln=True, zipf=1.5), name="train_ragged"),
        # The large model with a Zipf-skewed router: the largest training step.
        dict(_block("train", 32768, zipf=C3_ZIPF, **big), name="train_large"),
        # A large evaluation batch on MXFP4 experts packed once at load time.
        dict(_block("forward", 65536, 1024, 32, 4, 4096, weights="mxfp4_planes"), name="mxfp4_batch"),
        # The LayerNorm in front of the MLA block, forward and backward.
        {"kind": "norm", "T": 20480, "d": 1280, "name": "layernorm"},
        # The optimizer over one mid-sized block: LayerNorm, router, experts.
        {"kind": "adamw", "d": 512, "E": 8, "h": 2048, "clip": 1.0, "name": "adamw"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, odd=0.2):
    """A model or hidden width: mostly a multiple of 64, sometimes any number."""
    w = _log(rng, lo, hi)
    return w if rng.random() < odd else max(64, (w + 32) // 64 * 64)


def draw(rng):
    pick = rng.random()
    if pick < 0.08:
        return {"kind": "norm", "T": _log(rng, 64, 32768), "d": _width(rng, 128, 2560)}
    if pick < 0.16:
        return {"kind": "adamw", "d": _width(rng, 128, 1024, 0.3), "E": rng.randint(2, 16),
                "h": _width(rng, 256, 4096, 0.3), "clip": rng.choice((0.0, 1.0))}
    E = rng.choice((2, 4, 6, 8, 12, 16, 24, 32))
    K = min(E, rng.choice((1, 2, 2, 3, 4, 4, 6)))
    if pick < 0.40:  # decode
        quant = rng.random() < 0.3
        d, h = _width(rng, 256, 2048, 0.0 if quant else 0.1), _width(rng, 512, 4096, 0.0 if quant else 0.1)
        return _block("forward", _log(rng, 1, 64), d, E, K, h, weights="mxfp4" if quant else "bf16",
                      ln=not quant and rng.random() < 0.5)
    if pick < 0.60:  # prompts and evaluation batches
        quant = rng.random() < 0.4
        d, h = _width(rng, 256, 1280, 0.0 if quant else 0.2), _width(rng, 512, 4096, 0.0 if quant else 0.2)
        return _block("forward", _log(rng, 65, 16384), d, E, K, h,
                      weights=rng.choice(("mxfp4", "mxfp4_mx", "mxfp4_planes")) if quant else "bf16",
                      ln=not quant and rng.random() < 0.5, zipf=rng.choice((0.0, 1.0, 2.0)))
    # training; reference experts (h = 0) or up/down experts
    d = _width(rng, 128, 1280)
    h = 0 if rng.random() < 0.35 else _width(rng, 256, 4096)
    K = max(2, K)  # a renormalised top-1 gate is the constant 1: its router has no task gradient to train on
    return _block("train", _log(rng, 256, 16384), d, E, K, h, ln=rng.random() < 0.5, zipf=rng.choice((0.0, 1.0, 2.0)))


# ---- inputs ---------------------------------------------------------------

def _normal(gen, shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _inputs(case, seed):
    """The tensors a caller of the block has in hand, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T, d, E, h = case["T"], case["d"], case["E"], case["h"]
    hn = h if h > 0 else d
    t = {"X": _normal(gen, (T, d)), "dY": None}
    if case["ln"]:
        # a residual stream: rows of different scale and offset
        row = torch.rand((T, 2), generator=gen, device="cuda")
        t["X"] = (t["X"].float() * (0.5 + 2.0 * row[:, :1]) + (row[:, 1:] - 0.5)).to(torch.bfloat16)
        t["gamma"] = 1.0 + _normal(gen, (d,), 0.1, torch.float32)
        t["beta"] = _normal(gen, (d,), 0.1, torch.float32)
    t["Wr"] = _normal(gen, (E, d), d ** -0.5)
    t["W_up"] = torch.stack([_normal(gen, (hn, d), d ** -0.5) for _ in range(E)])
    t["W_down"] = torch.stack([_normal(gen, (d, h), h ** -0.5) for _ in range(E)]) if h > 0 else None
    t["bias"] = None
    if case["zipf"] > 0:
        t["bias"] = -case["zipf"] * torch.log(torch.arange(1, E + 1, device="cuda", dtype=torch.float32))
    if case["kind"] == "train":
        t["dY"] = _normal(gen, (T, d))
    return t


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _quantise(W):
    """bf16 [N, K] to MXFP4: codes [N, K/2] (low nibble = even column), scales
    [K/32, N] (e8m0); blocks of 32, scale exponent
    floor(log2 amax) - 2, nearest value, ties to the even code."""
    N, K = W.shape
    w = W.float().view(N, K // 32, 32)
    exp = torch.frexp(w.abs().amax(2))[1].int() - 3
    a = torch.ldexp(w.abs(), -exp[:, :, None])
    bounds = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=W.device)
    low, high = torch.bucketize(a, bounds), torch.bucketize(a, bounds, right=True)  # differ on a tie: the even code
    code = torch.where(low % 2 == 0, low, high).to(torch.uint8) | (torch.signbit(w).to(torch.uint8) << 3)
    code = code.view(N, K)
    return code[:, 0::2] | (code[:, 1::2] << 4), (exp + 127).to(torch.uint8).t().contiguous()


def _dequantise(codes, scales):
    """Exact values of _quantise's output, float64 [N, K]."""
    grid = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), device=codes.device, dtype=torch.float64)
    N = codes.shape[0]
    v = grid[torch.stack((codes & 15, codes >> 4), dim=2).long()].view(N, -1, 32)
    return torch.ldexp(v, scales.t().int()[:, :, None] - 127).view(N, -1)


def _quantised(W):
    """Stacked codes and scales of an expert weight tensor [E, N, K]."""
    both = [_quantise(w) for w in W]
    return torch.stack([b[0] for b in both]), torch.stack([b[1] for b in both])


def _norm_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    T, d = case["T"], case["d"]
    row = torch.rand((T, 2), generator=gen, device="cuda")
    S = torch.randn((T, d), generator=gen, device="cuda") * (0.5 + 2.0 * row[:, :1]) + (row[:, 1:] - 0.5)
    return {"S": S.to(torch.bfloat16), "dH": _normal(gen, (T, d)),
            "gamma": 1.0 + _normal(gen, (d,), 0.1, torch.float32), "beta": _normal(gen, (d,), 0.1, torch.float32)}


def _adamw_inputs(case, seed):
    """Parameters of one block after some updates: name -> fp32 master, moments
    and gradient; the experts are stacked [E, ...], as a caller keeps them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    d, E, h = case["d"], case["E"], case["h"]
    shapes = {"gamma": (1, d), "beta": (1, d), "Wr": (1, E, d), "W_up": (E, h, d), "W_down": (E, d, h)}
    out = {}
    for name, shape in shapes.items():
        # experts start at 16-byte boundaries, as the optimizer requires
        n = math.prod(shape[1:])
        full = (shape[0], (n + 3) // 4 * 4)
        std = shape[-1] ** -0.5
        make = lambda s: torch.randn(full, generator=gen, device="cuda")[:, :n] * s  # noqa: E731
        p = {k: torch.zeros(full, device="cuda") for k in ("master", "m", "v", "grad")}
        p["master"][:, :n] = make(std)
        p["m"][:, :n] = make(1e-3)
        p["v"][:, :n] = (make(1e-3) ** 2)
        p["grad"][:, :n] = make(2e-3)
        p["work"] = torch.zeros(shape[0], (n + 7) // 8 * 8, dtype=torch.bfloat16, device="cuda")
        p["work"][:, :n] = p["master"][:, :n].to(torch.bfloat16)
        p["n"] = n
        out[name] = p
    return out


_ADAMW = {"lr": 1e-3, "beta1": 0.9, "beta2": 0.999, "eps": 1e-8, "weight_decay": 0.01}
_ADAMW_STEP = 100  # updates done before the first measured one


def prepare(case, seed):
    """Inputs, weights, output buffers and the handle of a running program."""
    if case["kind"] == "norm":
        s = _norm_inputs(case, seed)
        T, d = case["T"], case["d"]
        s.update(case=case, H=torch.empty_like(s["S"]), mean=torch.empty(T, device="cuda"),
                 rstd=torch.empty(T, device="cuda"), dS=torch.empty_like(s["S"]),
                 dGamma=torch.empty(d, device="cuda"), dBeta=torch.empty(d, device="cuda"))
        s["workspace"] = torch.empty(max(tmt_moe.layernorm_workspace_size(T, d), 1), dtype=torch.uint8, device="cuda")
        return s
    if case["kind"] == "adamw":
        tensors = _adamw_inputs(case, seed)
        params = []
        for p in tensors.values():
            for e in range(p["master"].shape[0]):
                params.append({k: p[k][e, :p["n"]] for k in ("master", "m", "v", "grad", "work")})
        return {"case": case, "tensors": tensors, "opt": tmt_moe.AdamW(params), "step": _ADAMW_STEP}
    s = _inputs(case, seed)
    T, d, E, K, h = (case[k] for k in ("T", "d", "E", "K", "h"))
    fmt = case["weights"]
    if fmt != "bf16":
        for name in ("W_up", "W_down"):
            codes, scales = _quantised(s[name])
            if fmt == "mxfp4_planes":
                planes = torch.empty_like(codes)
                for e in range(E):
                    tmt_moe.mxfp4_planes(codes[e], planes[e])
                codes = planes
            s[name], s[name + "_scale"] = codes, scales
    s.update(case=case, moe=tmt_moe.MoE(T, d, E, K, h, weight_format=_FORMATS[fmt]), Y=torch.zeros_like(s["X"]))
    if case["kind"] == "train":
        s.update(dX=torch.empty_like(s["X"]), dWr=torch.empty(E, d, device="cuda"),
                 dW_up=torch.empty(s["W_up"].shape, device="cuda"),
                 dW_down=torch.empty(s["W_down"].shape, device="cuda") if h > 0 else None)
        if case["ln"]:
            s.update(dGamma=torch.empty(d, device="cuda"), dBeta=torch.empty(d, device="cuda"))
    return s


# TMT's aux and z-loss coefficients of the training configurations.
_AUX, _Z = 0.1, 1e-3


def run(s):
    case = s["case"]
    if case["kind"] == "norm":
        tmt_moe.layernorm_forward(s["S"], s["gamma"], s["beta"], s["H"], s["mean"], s["rstd"])
        tmt_moe.layernorm_backward(s["S"], s["dH"], s["gamma"], s["mean"], s["rstd"], s["dS"], s["dGamma"],
                                   s["dBeta"], s["workspace"])
        return {k: s[k] for k in ("H", "mean", "rstd", "dS", "dGamma", "dBeta")}
    if case["kind"] == "adamw":
        s["step"] += 1
        s["opt"].step(s["step"], clip=case["clip"], **_ADAMW)
        return {n: {k: p[k] for k in ("master", "m", "v", "work")} for n, p in s["tensors"].items()}
    moe, X, Wr, Wu, Wd, Y = (s[k] for k in ("moe", "X", "Wr", "W_up", "W_down", "Y"))
    if case["ln"]:
        Y.copy_(X)  # the residual stream: Y = X + MoE(LayerNorm(X))
        moe.forward_ln(X, s["gamma"], s["beta"], Wr, Wu, Wd, Y, beta=1.0, bias=s["bias"])
    elif case["weights"] == "bf16":
        moe.forward(X, Wr, Wu, Wd, Y, beta=0.0, bias=s["bias"])
    else:
        moe.forward_mxfp4(X, Wr, Wu, s["W_up_scale"], Wd, s["W_down_scale"], Y, beta=0.0, bias=s["bias"])
    if case["kind"] != "train":
        return {"Y": Y}
    out = {"Y": Y, "dX": s["dX"], "dWr": s["dWr"], "dW_up": s["dW_up"], "dW_down": s["dW_down"]}
    if case["ln"]:
        moe.backward_ln(s["dY"], X, s["gamma"], Wr, Wu, Wd, s["dX"], s["dGamma"], s["dBeta"], s["dWr"], s["dW_up"],
                        s["dW_down"], _AUX, _Z)
        out.update(dGamma=s["dGamma"], dBeta=s["dBeta"])
    else:
        moe.backward(s["dY"], X, Wr, Wu, Wd, s["dX"], s["dWr"], s["dW_up"], s["dW_down"], _AUX, _Z)
    return out


# ---- what a pass cannot do without -----------------------------------------

def work(case):
    if case["kind"] == "norm":
        T, d = case["T"], case["d"]
        # forward: S in, H out; backward: S and dH in, dS out; the row statistics out and in
        return {"bytes": 5 * 2 * T * d + 16 * T + 20 * d, "flops": 20 * T * d}
    if case["kind"] == "adamw":
        n = 2 * case["d"] + case["E"] * case["d"] * (1 + 2 * case["h"])
        return {"bytes": 30 * n, "flops": 15 * n}  # master, m, v, grad in; master, m, v and the bf16 copy out
    T, d, E, K, h = (case[k] for k in ("T", "d", "E", "K", "h"))
    mats, hn = (2, h) if h > 0 else (1, d)
    # experts that T * K independent picks reach on average; each one's weights are read once
    used = E * (1.0 - (1.0 - min(K, E) / E) ** T)
    per_weight = 2.0 if case["weights"] == "bf16" else 0.5 + 1.0 / 32
    nbytes = 2 * 2 * T * d + 2 * E * d + used * mats * hn * d * per_weight
    flops = 2.0 * T * d * E + 2.0 * mats * T * K * d * hn
    if case["ln"]:
        nbytes += 8 * d
    if case["kind"] == "train":
        # backward: dY, X and the weights in again, dX and the fp32 gradients out
        nbytes += 3 * 2 * T * d + used * mats * hn * d * 2 + 4 * (E * d + E * mats * hn * d)
        flops += 2 * (2.0 * T * d * E + 2.0 * mats * T * K * d * hn)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "norm":
        # dS: one rounding to bf16 (2^-9 / sqrt(3) = 1.1e-3), everything else is fp32
        return {"rel": 3e-3, "max": 2e-2}
    if case["kind"] == "adamw":
        # fp32 elementwise; the bf16 copy may round the other way at a tie (5e-5 of its values)
        return {"rel": 2e-5, "max": 1e-2}
    # Activations, hidden activations and expert outputs are rounded to bf16
    # between fp32-accumulating products: 2e-3 to 4e-3 against 64 bits.
    return {"rel": 1e-2, "max": 0.1}


# ---- the same in 64 bits ----------------------------------------------------

def _layernorm64(S, gamma, beta):
    x = S.double()
    mean = x.mean(1)
    var = ((x - mean[:, None]) ** 2).mean(1)
    rstd = (var + 1e-5).rsqrt()
    return ((x - mean[:, None]) * rstd[:, None]) * gamma.double() + beta.double(), mean, rstd


def _layernorm64_backward(S, g, gamma, mean, rstd):
    xh = (S.double() - mean[:, None]) * rstd[:, None]
    t = g * gamma.double()
    dS = rstd[:, None] * (t - t.mean(1, keepdim=True) - xh * (t * xh).mean(1, keepdim=True))
    return dS, (g * xh).sum(0), g.sum(0)


def exact(case, seed):
    if case["kind"] == "norm":
        s = _norm_inputs(case, seed)
        H, mean, rstd = _layernorm64(s["S"], s["gamma"], s["beta"])
        dS, dGamma, dBeta = _layernorm64_backward(s["S"], s["dH"].double(), s["gamma"], mean, rstd)
        return {"H": H, "mean": mean, "rstd": rstd, "dS": dS, "dGamma": dGamma, "dBeta": dBeta}
    if case["kind"] == "adamw":
        return _adamw64(case, seed)
    return _block64(case, seed)


def _adamw64(case, seed):
    t = _adamw_inputs(case, seed)
    total = sum((p["grad"].double() ** 2).sum() for p in t.values())
    scale = min(1.0, case["clip"] / max(math.sqrt(float(total)), 1e-12)) if case["clip"] > 0 else 1.0
    b1, b2, step = _ADAMW["beta1"], _ADAMW["beta2"], _ADAMW_STEP + 1
    out = {}
    for name, p in t.items():
        g = p["grad"].double() * scale
        m = b1 * p["m"].double() + (1 - b1) * g
        v = b2 * p["v"].double() + (1 - b2) * g * g
        w = p["master"].double()
        w = w - _ADAMW["lr"] * ((m / (1 - b1 ** step)) / ((v / (1 - b2 ** step)).sqrt() + _ADAMW["eps"])
                                + _ADAMW["weight_decay"] * w)
        work = torch.zeros(p["work"].shape, dtype=torch.float64, device="cuda")
        work[:, :p["n"]] = w[:, :p["n"]]
        out[name] = {"master": w, "m": m, "v": v, "work": work}
    return out


def _block64(case, seed):
    """The block by its formulas, expert by expert; gradients written out. The
    LayerNorm's output is rounded to bf16: it is the router's input by contract,
    and the picks depend on it."""
    s = _inputs(case, seed)
    T, d, E, K, h = (case[k] for k in ("T", "d", "E", "K", "h"))
    X = s["X"].double()
    if case["ln"]:
        H, mean, rstd = _layernorm64(s["X"], s["gamma"], s["beta"])
        H = H.to(torch.bfloat16).double()
    else:
        H = X

    def weights(name, e):
        W = s[name][e]
        return W.double() if case["weights"] == "bf16" else _dequantise(*_quantise(W))

    Wr = s["Wr"].double()
    logits = H @ Wr.t()
    if s["bias"] is not None:
        logits = logits + s["bias"].double()
    probs, lse = torch.softmax(logits, 1), torch.logsumexp(logits, 1)
    idx = torch.topk(logits, K, dim=1).indices
    psel = probs.gather(1, idx)
    gate = psel / psel.sum(1, keepdim=True)
    Y = X.clone() if case["ln"] else torch.zeros_like(X)
    train = case["kind"] == "train"
    if train:
        dY = s["dY"].double()
        dH, dgate = torch.zeros_like(X), torch.zeros_like(gate)
        dWu, dWd = [], []
    for e in range(E):
        rows, js = torch.nonzero(idx == e, as_tuple=True)
        Wu = weights("W_up", e)
        u = H[rows] @ Wu.t()
        sg = torch.sigmoid(u)
        a = u * sg
        Wd = weights("W_down", e) if h > 0 else None
        o = a @ Wd.t() if h > 0 else a
        g = gate[rows, js][:, None]
        Y.index_add_(0, rows, g * o)
        if train:
            dgate[rows, js] = (dY[rows] * o).sum(1)
            do = g * dY[rows]
            da = do @ Wd if h > 0 else do
            du = da * (sg * (1 + u * (1 - sg)))
            dWu.append(du.t() @ H[rows])
            if h > 0:
                dWd.append(do.t() @ a)
            dH.index_add_(0, rows, du @ Wu)
    if not train:
        return {"Y": Y}
    # router: renormalised gates, softmax, aux (expert fractions constant), z
    dpsel = (dgate - (dgate * gate).sum(1, keepdim=True)) / psel.sum(1, keepdim=True)
    frac = torch.bincount(idx.reshape(-1), minlength=E).double() / (T * K)
    dprobs = torch.zeros_like(probs).scatter_(1, idx, dpsel) + _AUX * E * frac / T
    dlogits = probs * (dprobs - (dprobs * probs).sum(1, keepdim=True)) + (2 * _Z / T) * lse[:, None] * probs
    dH += dlogits @ Wr
    out = {"Y": Y, "dX": dH, "dWr": dlogits.t() @ H, "dW_up": torch.stack(dWu),
           "dW_down": torch.stack(dWd) if h > 0 else None}
    if case["ln"]:
        out["dX"], out["dGamma"], out["dBeta"] = _layernorm64_backward(s["X"], dH, s["gamma"], mean, rstd)
    return out
