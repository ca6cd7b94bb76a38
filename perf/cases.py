"""The calls that the performance of this framework is judged by.

Each case is one pass of work through a public entry point, on inputs made from a
seed: the standalone scans (``kla.ops.hip.mobius_scan``, ``affine_scan``), the KLA
scan (``kla.kla_scan``), one ``KLALayer`` (inference with and without a carried
state, and a training step) and a ``SequenceModel`` (prefill and one-token decode).
``listed`` names the representative ones; ``draw`` gives others of the same ranges.
``exact`` restates every path step by step in float64 torch.

Values are those the layer hands on in use: decays exp(-Delta) with Delta between
1e-3 and 1e-1, Ornstein-Uhlenbeck process noise, precisions 1 / softplus, l2-normed
k and q, weights at the scale of their initialisation with the static parameters
moved off their constant start.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "kalman-linear-attention_amd"))

from kla import KLAConfig, KLALayer, KLALayerState, KLAState, ModelConfig, SequenceModel, kla_scan  # noqa: E402
from kla.models.decode_graph import DecodeGraph  # noqa: E402
from kla.ops.hip import affine_scan, mobius_scan  # noqa: E402

DEV = "cuda"
EPS = 1e-12
VOCAB = 50304


def listed():
    return [
        # A unit-test sized scan: launches and look-back latency are all of it.
        {"name": "mobius_small", "kind": "mobius", "B": 2, "T": 300, "lanes": 130, "D": True},
        # The headline workload's precision scan, forward and backward.
        {"name": "mobius_headline", "kind": "mobius", "B": 8, "T": 4096, "lanes": 2048, "D": False},
        # A general first-order recurrence between them: odd sizes, an initial state, fp32.
        {"name": "affine_ragged", "kind": "affine", "B": 3, "T": 2501, "lanes": 1100, "dtype": "f32", "h0": True},
        # The long bf16 scan of the benchmark.
        {"name": "affine_bf16_long", "kind": "affine", "B": 8, "T": 8192, "lanes": 2048, "dtype": "bf16", "h0": False},
        # One prompt of odd length through the filter with a carried state (serving).
        {"name": "kla_infer_ragged", "kind": "kla", "B": 1, "L": 1021, "M": 1024, "S": 16, "train": False,
         "state": True},
        # Training the filter alone at a wide state.
        {"name": "kla_train_state128", "kind": "kla", "B": 2, "L": 2048, "M": 512, "S": 128, "train": True,
         "state": False},
        # The benchmark's layer forward, fp32 inference without a state.
        {"name": "layer_forward", "kind": "layer", "d": 512, "B": 2, "L": 1024, "block": "plain", "mode": "infer",
         "dtype": "f32", "state": False},
        # A prefill chunk of odd length through a wide layer that carries its state.
        {"name": "layer_prefill_ragged", "kind": "layer", "d": 1024, "B": 4, "L": 2047, "block": "plain",
         "mode": "infer", "dtype": "f32", "state": True},
        # The benchmark's training step: bf16 autocast, 16384 tokens.
        {"name": "layer_train_bf16", "kind": "layer", "d": 1024, "B": 4, "L": 4096, "block": "plain", "mode": "train",
         "dtype": "bf16", "state": False},
        # A small fp32 training step with low-rank sensors (value from the conv, variance of rank d/8).
        {"name": "layer_train_small", "kind": "layer", "d": 384, "B": 2, "L": 500, "block": "lowrank",
         "mode": "train", "dtype": "f32", "state": False},
        # The default model's prefill of four prompts, to logits at every position.
        {"name": "model_prefill", "kind": "prefill", "layers": 6, "B": 4, "L": 1024},
        # One token for each of 16 sequences by the replayed decode graph.
        {"name": "model_decode", "kind": "decode", "layers": 6, "B": 16, "L": 48},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sizes(rng, ranges, most, least=1):
    """Integers spread over the logarithm of each (lo, hi), their product between ``least`` and ``most``."""
    while True:
        got = [_log_int(rng, lo, hi) for lo, hi in ranges]
        if least <= math.prod(got) <= most:
            return got


def draw(rng):
    kind = rng.choice(("mobius", "affine", "kla", "kla", "layer", "layer", "layer", "prefill", "decode"))
    if kind == "mobius":
        B, T, lanes = _sizes(rng, ((1, 16), (64, 8192), (32, 4096)), 1 << 26, 1 << 14)
        return {"kind": kind, "B": B, "T": T, "lanes": lanes, "D": rng.random() < 0.25}
    if kind == "affine":
        B, T, lanes = _sizes(rng, ((1, 16), (64, 8192), (32, 4096)), 1 << 27, 1 << 14)
        return {"kind": kind, "B": B, "T": T, "lanes": lanes, "dtype": rng.choice(("f32", "bf16")),
                "h0": rng.random() < 0.5}
    if kind == "kla":
        S = rng.choice((4, 8, 16, 16, 16, 24, 32, 64, 128, 200, 256))
        B, L, M = _sizes(rng, ((1, 16), (64, 4096), (64, 2048)), (1 << 28) // S, 1 << 14)
        return {"kind": kind, "B": B, "L": L, "M": M, "S": S, "train": rng.random() < 0.5,
                "state": rng.random() < 0.5}
    if kind == "layer":
        d = rng.choice((256, 384, 512, 768, 1024))
        mode = rng.choice(("infer", "infer", "train"))
        B, L = _sizes(rng, ((1, 16), (64, 4096)), (1 << 24) // d, 256)
        return {"kind": kind, "d": d, "B": B, "L": L, "block": rng.choice(("plain", "plain", "lowrank")),
                "mode": mode, "dtype": rng.choice(("f32", "bf16")),
                "state": mode == "infer" and rng.random() < 0.5}
    if kind == "prefill":
        B, L = _sizes(rng, ((1, 4), (64, 1024)), 4096, 64)
        return {"kind": kind, "layers": rng.choice((2, 4, 6)), "B": B, "L": L}
    return {"kind": "decode", "layers": rng.choice((2, 4, 6)), "B": _log_int(rng, 1, 64), "L": _log_int(rng, 16, 64)}


# ------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _scan_inputs(case, seed):
    g = _gen(seed)
    shape = (case["B"], case["T"], case["lanes"])
    state = (case["B"], case["lanes"])

    def rn(*s):
        return torch.randn(*s, device=DEV, generator=g)

    if case["kind"] == "mobius":
        ins = {"A": torch.exp(-F.softplus(rn(*shape))), "B": F.softplus(rn(*shape)), "C": F.softplus(rn(*shape)),
               "D": F.softplus(rn(*shape)) + 0.5 if case["D"] else None, "lam0": F.softplus(rn(*state)),
               "dout": rn(*shape)}
    else:
        dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        ins = {"g": torch.sigmoid(rn(*shape)).to(dt), "u": rn(*shape).to(dt),
               "h0": rn(*state) if case["h0"] else None, "dout": rn(*shape).to(dt)}
    return ins


def _dynamics(M, S, g):
    """Discrete (a, p) as a layer with Delta in [1e-3, 1e-1], rates near 1 and process noise near 0.01 has them."""
    delta = torch.exp(math.log(1e-3) + math.log(100.0) * torch.rand(M, S, device=DEV, generator=g))
    rate = torch.exp(0.2 * torch.randn(M, S, device=DEV, generator=g))
    noise = 0.01 * torch.exp(0.2 * torch.randn(M, S, device=DEV, generator=g))
    return torch.exp(-delta * rate), noise / (2 * rate) * -torch.expm1(-2 * rate * delta)


def _kla_inputs(case, seed):
    g = _gen(seed)
    B, L, M, S = (case[n] for n in ("B", "L", "M", "S"))

    def rn(*s):
        return torch.randn(*s, device=DEV, generator=g)

    a, p = _dynamics(M, S, g)
    ins = {"v": rn(B, L, M), "lambda_v": 1.0 / (F.softplus(rn(B, L, M)) + 1e-4),
           "k": F.normalize(rn(B, L, S), dim=-1), "q": F.normalize(rn(B, L, S), dim=-1), "a": a, "p": p,
           "lam0": None, "eta0": None}
    if case["state"]:
        ins["lam0"], ins["eta0"] = F.softplus(rn(B, M, S)) + 0.5, rn(B, M, S)
    if case["train"]:
        ins["dy"], ins["dyv"] = rn(B, L, M), rn(B, L, M)
    return ins


def _layer_config(case):
    low = case.get("block") == "lowrank"
    return KLAConfig(value_rank="conv" if low else "full", var_rank="dt" if low else "full")


def _layer_weights(d, low, g, std=None):
    """A KLALayer's parameters by name; Linear weights at their fan-in scale, or ``std``."""
    M, S = 2 * d, 16
    rank = math.ceil(d / 8)

    def lin(out, inp):
        return torch.randn(out, inp, device=DEV, generator=g) * (1 / math.sqrt(3 * inp) if std is None else std)

    w = {"in_proj.weight": lin(2 * M, d),
         "conv.weight": torch.randn(M, 1, 4, device=DEV, generator=g) * 0.3,
         "conv.bias": torch.randn(M, device=DEV, generator=g) * 0.02,
         "sensor_proj.weight": lin((rank if low else 2 * M) + 2 * S, M)}
    if low:
        w["var_expand.weight"] = lin(M, rank)
    delta = torch.exp(math.log(1e-3) + math.log(100.0) * torch.rand(M, S, device=DEV, generator=g))
    w["delta"] = delta + torch.log(-torch.expm1(-delta))
    w["lambda_log"] = 0.2 * torch.randn(M, S, device=DEV, generator=g)
    w["process_noise"] = 0.01 * torch.exp(0.2 * torch.randn(M, S, device=DEV, generator=g))
    w["lambda_skip"] = torch.tensor(-1.0, device=DEV)
    w["out_proj.weight"] = lin(d, M)
    return w


def _layer_state(d, B, g):
    """(conv window, lam, eta) as an earlier chunk leaves them."""
    return (torch.randn(B, 2 * d, 3, device=DEV, generator=g) * 0.5,
            1.0 + 20.0 * torch.rand(B, 2 * d, 16, device=DEV, generator=g),
            torch.randn(B, 2 * d, 16, device=DEV, generator=g) * 3.0)


def _layer_inputs(case, seed):
    g = _gen(seed)
    w = _layer_weights(case["d"], case["block"] == "lowrank", g)
    x = torch.randn(case["B"], case["L"], case["d"], device=DEV, generator=g)
    dout = (torch.randn(case["B"], case["L"], case["d"], device=DEV, generator=g)
            if case["mode"] == "train" else None)
    return w, x, dout, _layer_state(case["d"], case["B"], g) if case["state"] else None


def _model_inputs(case, seed):
    g = _gen(seed)
    d, hidden = 512, int(2 * 2048 / 3)
    w = {"embedding.weight": torch.randn(VOCAB, d, device=DEV, generator=g),
         "lm_head.weight": torch.randn(VOCAB, d, device=DEV, generator=g) * 0.02,
         "norm_f.weight": 1 + 0.1 * torch.randn(d, device=DEV, generator=g)}
    for i in range(case["layers"]):
        for name, t in _layer_weights(d, False, g, std=0.02).items():
            w[f"blocks.{i}.mixer.{name}"] = t
        for norm in ("mixer_norm", "mlp_norm"):
            w[f"blocks.{i}.{norm}.weight"] = 1 + 0.1 * torch.randn(d, device=DEV, generator=g)
        w[f"blocks.{i}.mlp.w12.weight"] = torch.randn(2 * hidden, d, device=DEV, generator=g) * 0.02
        w[f"blocks.{i}.mlp.w3.weight"] = torch.randn(d, hidden, device=DEV, generator=g) * 0.02
    ids = torch.randint(0, VOCAB, (case["B"], case["L"]), device=DEV, generator=g)
    token = torch.randint(0, VOCAB, (case["B"], 1), device=DEV, generator=g)
    return w, ids, token


# ------------------------------------------------------------ prepare and run


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("mobius", "affine"):
        ins = _scan_inputs(case, seed)
        dout = ins.pop("dout")
        return {"kind": kind, "dout": dout,
                "ins": {n: None if t is None else t.requires_grad_(True) for n, t in ins.items()}}
    if kind == "kla":
        ins = _kla_inputs(case, seed)
        grads = [ins.pop(n) for n in ("dy", "dyv")] if case["train"] else None
        if case["train"]:
            ins = {n: None if t is None else t.requires_grad_(True) for n, t in ins.items()}
        return {"kind": kind, "ins": ins, "grads": grads}
    if kind == "layer":
        w, x, dout, st = _layer_inputs(case, seed)
        with torch.device(DEV):
            layer = KLALayer(case["d"], _layer_config(case))
        layer.load_state_dict(w)
        train = case["mode"] == "train"
        layer.train(train)
        state = None
        if st is not None:
            state = KLALayerState(conv=st[0], ssm=KLAState(lam=st[1], eta=st[2]))
        return {"kind": kind, "layer": layer, "x": x.requires_grad_(train), "dout": dout, "state": state,
                "bf16": case["dtype"] == "bf16", "train": train}
    w, ids, token = _model_inputs(case, seed)
    with torch.device(DEV):
        model = SequenceModel(ModelConfig(vocab_size=VOCAB, d_model=512, n_layers=case["layers"]), KLAConfig()).eval()
    model.load_state_dict(w)
    if kind == "prefill":
        return {"kind": kind, "model": model, "ids": ids}
    with torch.no_grad():
        _, state = model(ids, state=model.init_state(case["B"]))
    return {"kind": kind, "graph": DecodeGraph(model, state), "token": token}


def _flat_state(states):
    return [t for s in states for t in (s.conv, s.ssm.lam, s.ssm.eta)]


def run(state):
    kind = state["kind"]
    if kind in ("mobius", "affine"):
        ins = state["ins"]
        out = mobius_scan(**ins) if kind == "mobius" else affine_scan(**ins)
        wrt = [t for t in ins.values() if t is not None]
        return [out.detach(), *torch.autograd.grad(out, wrt, state["dout"])]
    if kind == "kla":
        ins = state["ins"]
        st = None if ins["lam0"] is None else KLAState(lam=ins["lam0"], eta=ins["eta0"])
        args = (ins["v"], ins["lambda_v"], ins["k"], ins["q"], ins["a"], ins["p"])
        if state["grads"] is None:
            with torch.no_grad():
                y, y_var, fin = kla_scan(*args, initial_state=st)
            return [y, y_var, fin.lam, fin.eta]
        y, y_var, fin = kla_scan(*args, initial_state=st)
        wrt = [t for t in ins.values() if t is not None]
        return [y.detach(), y_var.detach(), fin.lam.detach(), fin.eta.detach(),
                *torch.autograd.grad((y, y_var), wrt, state["grads"])]
    if kind == "layer":
        layer, x = state["layer"], state["x"]
        if not state["train"]:
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=state["bf16"]):
                out, new = layer(x, state["state"], return_state=True)
            return [out, *_flat_state([new])]
        layer.zero_grad(set_to_none=True)
        x.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=state["bf16"]):
            out = layer(x)
        out.backward(state["dout"].to(out.dtype))
        return [out.detach(), x.grad, *(p.grad for _, p in sorted(layer.named_parameters()))]
    if kind == "prefill":
        model = state["model"]
        with torch.no_grad():
            logits, new = model(state["ids"], state=model.init_state(state["ids"].shape[0]))
        return [logits, *_flat_state(new)]
    logits = state["graph"].step(state["token"])
    return [logits, *_flat_state(state["graph"].state)]


# ------------------------------------------------------------------- work


def _layer_sizes(d, low):
    """(weights in the projections, all parameters) of a KLALayer."""
    M, S, rank = 2 * d, 16, math.ceil(d / 8)
    mat = 2 * M * d + ((rank if low else 2 * M) + 2 * S) * M + (M * rank if low else 0) + d * M
    return mat, mat + 5 * M + 3 * M * S + 1


def work(case):
    kind = case["kind"]
    if kind == "mobius":
        n = case["B"] * case["T"] * case["lanes"]
        # A, B, C (D) and the gradient in; lam and the gradients out.
        return {"bytes": n * 4.0 * (8 + 2 * case["D"]), "flops": 20.0 * n}
    if kind == "affine":
        n = case["B"] * case["T"] * case["lanes"]
        return {"bytes": n * 6.0 * (2 if case["dtype"] == "bf16" else 4), "flops": 6.0 * n}
    if kind == "kla":
        B, L, M, S = (case[n] for n in ("B", "L", "M", "S"))
        seq, row, st = B * L * M, B * L * S, B * M * S
        bytes_ = 4.0 * (4 * seq + 2 * row + 2 * M * S + st * (4 if case["state"] else 2))
        if case["train"]:
            bytes_ += 4.0 * (4 * seq + 2 * row + 2 * M * S + (2 * st if case["state"] else 0))
        return {"bytes": bytes_, "flops": (45.0 if case["train"] else 15.0) * seq * S}
    if kind == "layer":
        mat, params = _layer_sizes(case["d"], case["block"] == "lowrank")
        tok = case["B"] * case["L"]
        lane_steps = tok * 2 * case["d"] * 16
        state = 2 * case["B"] * 2 * case["d"] * 35 if case["state"] else case["B"] * 2 * case["d"] * 35
        out = 2.0 if case["dtype"] == "bf16" else 4.0
        if case["mode"] == "infer":
            return {"bytes": 4.0 * (tok * case["d"] + params + state) + out * tok * case["d"],
                    "flops": 2.0 * mat * tok + 15.0 * lane_steps}
        return {"bytes": 4.0 * (2 * tok * case["d"] + 2 * params) + (out + 4.0) * tok * case["d"],
                "flops": 6.0 * mat * tok + 45.0 * lane_steps}
    d, hidden = 512, int(2 * 2048 / 3)
    mat, params = _layer_sizes(d, False)
    mat, params = mat + 3 * hidden * d, params + 3 * hidden * d + 2 * d
    tok = case["B"] * (case["L"] if kind == "prefill" else 1)
    weights = case["layers"] * params + VOCAB * d + d
    state = case["layers"] * case["B"] * 2 * d * 35 * (1 if kind == "prefill" else 2)
    return {"bytes": 4.0 * (weights + tok * d + state + tok * VOCAB) + 8.0 * tok,
            "flops": 2.0 * tok * (case["layers"] * mat + VOCAB * d) + 15.0 * tok * case["layers"] * 2 * d * 16}


def tolerance(case):
    kind = case["kind"]
    if kind == "affine" and case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.1}
    if kind in ("mobius", "affine"):
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "layer" and case["dtype"] == "bf16":
        return {"rel": 3e-2, "max": 0.5}
    if kind in ("prefill", "decode"):
        return {"rel": 5e-5, "max": 2e-3}
    return {"rel": 3e-5, "max": 2e-3}


# ------------------------------------------------------------------- exact


def _exact_mobius(ins):
    A, B, C, D, lam0, dout = (None if ins[n] is None else ins[n].double() for n in ("A", "B", "C", "D", "lam0", "dout"))
    T = A.shape[1]
    lam, prev = torch.empty_like(A), torch.empty_like(A)
    x = lam0
    for t in range(T):
        prev[:, t] = x
        x = (A[:, t] * x + B[:, t]) / (C[:, t] * x + (1.0 if D is None else D[:, t]))
        lam[:, t] = x
    inv = 1.0 / (C * prev + (1.0 if D is None else D))
    gain = (A - lam * C) * inv
    nu, g = torch.empty_like(A), torch.zeros_like(lam0)
    for t in reversed(range(T)):
        nu[:, t] = dout[:, t] + g
        g = gain[:, t] * nu[:, t]
    nu *= inv
    out = [lam, nu * prev, nu, -nu * lam * prev]
    return out + ([] if D is None else [-nu * lam]) + [g]


def _exact_affine(ins):
    g, u, dout = (ins[n].double() for n in ("g", "u", "dout"))
    h0 = None if ins["h0"] is None else ins["h0"].double()
    T = g.shape[1]
    h, prev = torch.empty_like(g), torch.empty_like(g)
    x = torch.zeros_like(g[:, 0]) if h0 is None else h0
    for t in range(T):
        prev[:, t] = x
        x = g[:, t] * x + u[:, t]
        h[:, t] = x
    du, w = torch.empty_like(g), torch.zeros_like(x)
    for t in reversed(range(T)):
        du[:, t] = dout[:, t] + w
        w = g[:, t] * du[:, t]
    return [h, du * prev, du] + ([] if h0 is None else [w])


class _Filter(torch.autograd.Function):
    """The filter step by step, (phi, r [B, L, M, S], a, p [M, S], lam0, eta0 [B, M, S]) -> lam, eta at every
    step, with its adjoint step by step. All float64."""

    @staticmethod
    def forward(ctx, phi, r, a, p, lam0, eta0):
        lam, eta = torch.empty_like(phi), torch.empty_like(r)
        x, e, a2 = lam0, eta0, a * a
        for t in range(phi.shape[1]):
            den = torch.addcmul(a2, p, x)
            x = x / den + phi[:, t]
            e = a * e / den + r[:, t]
            lam[:, t], eta[:, t] = x, e
        ctx.save_for_backward(a, p, lam0, eta0, lam, eta)
        return lam, eta

    @staticmethod
    def backward(ctx, dlam, deta):
        a, p, lam0, eta0, lam, eta = ctx.saved_tensors
        dphi, dr = torch.empty_like(lam), torch.empty_like(eta)
        gl, ge, a2 = torch.zeros_like(lam0), torch.zeros_like(eta0), a * a
        da, dp = torch.zeros_like(lam0), torch.zeros_like(lam0)
        for t in reversed(range(lam.shape[1])):
            x, e = (lam0, eta0) if t == 0 else (lam[:, t - 1], eta[:, t - 1])
            gl, ge = gl + dlam[:, t], ge + deta[:, t]
            dphi[:, t], dr[:, t] = gl, ge
            inv = 1.0 / torch.addcmul(a2, p, x)
            dden = -(gl * x + ge * a * e) * inv * inv
            da += ge * e * inv + 2 * a * dden
            dp += dden * x
            gl, ge = gl * inv + dden * p, ge * a * inv
        return dphi, dr, da.sum(0), dp.sum(0), gl, ge


def _filter(v, lv, k, q, a, p, lam0, eta0):
    """(y, y_var, lam, eta at the end) in float64."""
    B, _, M = v.shape
    S = k.shape[-1]
    lam0 = v.new_ones(B, M, S) if lam0 is None else lam0
    eta0 = v.new_zeros(B, M, S) if eta0 is None else eta0
    lam, eta = _Filter.apply(lv.unsqueeze(-1) * (k * k).unsqueeze(-2), (v * lv).unsqueeze(-1) * k.unsqueeze(-2), a, p,
                             lam0, eta0)
    qs = q.unsqueeze(-2)
    var = 1.0 / lam
    return (eta * var * qs).sum(-1), (var * (qs * qs)).sum(-1), lam[:, -1], eta[:, -1]


def _exact_kla(case, ins):
    names = [n for n in ("v", "lambda_v", "k", "q", "a", "p", "lam0", "eta0") if ins[n] is not None]
    xs = {n: ins[n].double().requires_grad_(case["train"]) for n in names}
    outs = _filter(*(xs.get(n) for n in ("v", "lambda_v", "k", "q", "a", "p", "lam0", "eta0")))
    if not case["train"]:
        return list(outs)
    grads = torch.autograd.grad(outs[:2], [xs[n] for n in names], [ins["dy"].double(), ins["dyv"].double()])
    return [*(t.detach() for t in outs), *grads]


def _exact_layer_forward(w, x, low, st):
    """A KLALayer's output and its new (conv, lam, eta), all float64."""
    M, S = w["in_proj.weight"].shape[0] // 2, 16
    z, gate = F.linear(x, w["in_proj.weight"]).split(M, dim=-1)
    window = x.new_zeros(x.shape[0], M, 3) if st is None else st[0]
    padded = torch.cat((window, z.transpose(1, 2)), dim=-1)
    taps, L = w["conv.weight"][:, 0], x.shape[1]
    z = sum(padded[..., j:j + L] * taps[:, j, None] for j in range(4)) + w["conv.bias"][:, None]
    z = F.silu(z).transpose(1, 2)
    proj = F.linear(z, w["sensor_proj.weight"])
    if low:
        code, k, q = proj.split([proj.shape[-1] - 2 * S, S, S], dim=-1)
        v, log_var = z, F.linear(code, w["var_expand.weight"])
    else:
        v, log_var, k, q = proj.split([M, M, S, S], dim=-1)
    lv = 1.0 / (F.softplus(log_var) + 1e-4)
    k, q = F.normalize(k, dim=-1, eps=EPS), F.normalize(q, dim=-1, eps=EPS)
    rate = torch.exp(w["lambda_log"])
    delta = F.softplus(w["delta"]) + 1e-7
    a, p = torch.exp(-delta * rate), w["process_noise"] / (2 * rate) * -torch.expm1(-2 * rate * delta)
    y, _, lam, eta = _filter(v, lv, k, q, a, p, None if st is None else st[1], None if st is None else st[2])
    out = F.linear((y + w["lambda_skip"] * z) * F.silu(gate), w["out_proj.weight"])
    return out, [padded[..., L:], lam, eta]


def _exact_layer(case, seed):
    w, x, dout, st = _layer_inputs(case, seed)
    train = case["mode"] == "train"
    w = {n: t.double().requires_grad_(train) for n, t in w.items()}
    x = x.double().requires_grad_(train)
    st = None if st is None else [t.double() for t in st]
    out, new = _exact_layer_forward(w, x, case["block"] == "lowrank", st)
    if not train:
        return [out, *new]
    names = sorted(w)
    grads = torch.autograd.grad(out, [x, *(w[n] for n in names)], dout.double())
    return [out.detach(), *grads]


def _exact_model(case, w, ids):
    w = {n: t.double() for n, t in w.items()}

    def norm(x, weight):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * weight

    x, states = w["embedding.weight"][ids], []
    for i in range(case["layers"]):
        pre = f"blocks.{i}."
        mixer = {n[len(pre) + 6:]: t for n, t in w.items() if n.startswith(pre + "mixer.")}
        y, new = _exact_layer_forward(mixer, norm(x, w[pre + "mixer_norm.weight"]), False, None)
        x = x + y
        h = F.linear(norm(x, w[pre + "mlp_norm.weight"]), w[pre + "mlp.w12.weight"])
        gate, up = h.chunk(2, dim=-1)
        x = x + F.linear(F.silu(gate) * up, w[pre + "mlp.w3.weight"])
        states += new
    if case["kind"] == "decode":
        x = x[:, -1:]
    return [F.linear(norm(x, w["norm_f.weight"]), w["lm_head.weight"]), *states]


def exact(case, seed):
    kind = case["kind"]
    if kind == "mobius":
        return _exact_mobius(_scan_inputs(case, seed))
    if kind == "affine":
        return _exact_affine(_scan_inputs(case, seed))
    if kind == "kla":
        return _exact_kla(case, _kla_inputs(case, seed))
    if kind == "layer":
        return _exact_layer(case, seed)
    w, ids, token = _model_inputs(case, seed)
    return _exact_model(case, w, ids if kind == "prefill" else torch.cat((ids, token), dim=1))
