"""The calls whose speed matters to a user of this package, with their inputs and results.

Every case goes through a public entry point (``DABSNCore``, ``DABSNRead``, ``DABSNBlock``,
``DABSNSequenceLM``, ``forward_with_memory``, the losses and the registered operators) with
sizes of the package's own configurations:

  scan    the core recurrence of one layer, forward and backward
  read    the memory read of one layer: seq, field or hybrid, training or evaluation
  long    the recurrent long-memory channel, forward and backward
  delta   the permanent delta scan, forward and backward
  loss    the readout with its chunked cross-entropy, forward and backward
  block   a whole seq block with time chunking (the wide single-layer language model)
  lm      one training step of a small language model
  decode  one token of streaming decode against a carried memory

``exact`` evaluates the same expressions in 64 bits with plain tensor operations.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import dabsn_amd
from dabsn_amd import kernels

DEVICE = "cuda"

#: Initial values of the parameters that do not start from a random matrix (core.py, read.py,
#: model.py); a case adds a spread to them, as training does. The write gate's bias starts from
#: -2 and rises as the layer learns to write: -1 here.
BASE = {
    "logit_alpha": -2.0, "log_lambda": -1.0, "log_kappa": -2.25, "logit_recover": -4.6,
    "logit_saturation_decay": 2.2, "logit_saturation_suppress": -6.0, "Wg.bias": -1.0,
    "log_temp": 0.0, "p_gain": 1.0, "novelty_gain": 0.5, "null_bias": -2.0, "adm_p_gain": 1.0,
    "adm_novelty_gain": 0.5, "adm_saturation_gain": 0.5, "adm_energy_gain": 0.25,
    "adm_bias": -2.0, "pad_gain": 1.0, "short_gain": 1.0, "induct_gain": 0.1,
    "cocktail_gain": 1.0, "hybrid_gate": 0.0, "admit_window": 4.0, "logit_retain": 2.2,
    "long_gain": 0.1, "logit_expect_retain": 2.2, "logit_retention_decay": 2.2,
    "logit_retention_strength": 1.4, "read_gain": 0.1, "mlp_norm.weight": 1.0,
}

#: These shift every score of a softmax alike: their gradients are zero up to rounding, and
#: the selection window has none, so a program gains nothing by asking for them.
FROZEN = ("null_bias", "adm_bias", "admit_window")


def listed():
    return [
        # The quick-start model's first layer (state 96, input 24, batch 8, 256 steps): a call
        # where latency is all there is.
        dict(name="scan_quickstart", kind="scan", dtype="fp32", B=8, T=256, D=24, H=96),
        # The group-tracking language model's layer at its training length.
        dict(name="scan_tracking", kind="scan", dtype="fp32", B=16, T=256, D=512, H=512),
        # One time chunk of the wide single-layer language model, bf16 activations.
        dict(name="scan_wide", kind="scan", dtype="bf16", B=16, T=1024, D=2048, H=2048),
        # The read of the same layer over a training sequence.
        dict(name="read_wide", kind="read", dtype="bf16", B=16, T=1024, H=2048, geometry="seq",
             train=True),
        # The copy task's evaluation length (3,200 tokens, batch 32, state 256).
        dict(name="read_copy_eval", kind="read", dtype="fp32", B=32, T=3200, H=256,
             geometry="seq", train=False),
        # A hybrid read (causal and whole-sequence) over a ragged field, in training.
        dict(name="read_hybrid", kind="read", dtype="fp32", B=8, T=577, H=192,
             geometry="hybrid", train=True),
        # The long-memory channel of the wide layer over its whole sequence.
        dict(name="long_wide", kind="long", dtype="bf16", B=16, T=4096, H=2048),
        # The permanent associative primitive.
        dict(name="delta", kind="delta", dtype="fp32", B=16, T=1024, H=256),
        # Readout and loss of a 32,000-word vocabulary over 8,192 tokens.
        dict(name="loss_wide", kind="loss", dtype="bf16", N=8192, V=32000, H=2048),
        # The benchmark's layer as a block: projections, chunked scan, read, long channel.
        dict(name="block_wide", kind="block", dtype="bf16", B=16, T=4096, D=4096, H=2048,
             chunk=1024),
        # A training step of the copy-task model: 64 tokens, two layers, launches dominate.
        dict(name="lm_copy_step", kind="lm", dtype="fp32", B=32, T=64, H=256, layers=2, V=65),
        # Streaming decode: one token for each of 256 sequences after a 2,048-token prompt.
        dict(name="decode", kind="decode", dtype="bf16", B=256, H=2048, layers=4, prompt=2048,
             V=32000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, step):
    """A state width: mostly a multiple of ``step``, sometimes any number."""
    h = _log(rng, lo, hi)
    return h if rng.random() < 0.2 and h < 1024 else max(step, h // step * step)


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "read", "read", "read", "long", "delta", "loss",
                       "block", "lm", "decode"])
    dtype = rng.choice(["fp32", "bf16"])
    if kind == "scan":
        H = _width(rng, 64, 2048, 16)
        T = _log(rng, 16, 1024)
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 32 if H <= 1024 else 16), T=T,
                    D=_log(rng, 16, 1024) // 8 * 8, H=H)
    if kind == "read":
        H = _width(rng, 64, 2048, 16)
        T = _log(rng, 32, 3200)
        top = max(1, min(32, int(1.5e8 / (T * H)), int(3e8 / (T * T))))
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, top), T=T, H=H,
                    geometry=rng.choice(["seq", "seq", "seq", "field", "hybrid"]),
                    train=rng.random() < 0.7)
    if kind == "long":
        H = _width(rng, 64, 2048, 16)
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 16), T=_log(rng, 32, 4096), H=H)
    if kind == "delta":
        return dict(kind=kind, dtype=dtype, B=rng.randint(1, 16), T=_log(rng, 16, 1024),
                    H=_width(rng, 32, 256, 8))
    if kind == "loss":
        # fp32 models are the narrow ones
        H = _width(rng, 64, 2048 if dtype == "bf16" else 512, 8)
        V = _log(rng, 60, 32000)
        return dict(kind=kind, dtype=dtype, N=max(16, min(_log(rng, 256, 16384), int(2e8 / V))),
                    V=V, H=H)
    if kind == "block":
        T = rng.choice([768, 1024, 1536, 2048])
        H = rng.choice([1024, 1536, 2048])
        return dict(kind=kind, dtype="bf16", B=rng.choice([8, 12, 16]), T=T,
                    D=rng.choice([1024, 2048, 4096]), H=H, chunk=rng.choice([256, 512]))
    if kind == "lm":
        return dict(kind=kind, dtype="fp32", B=rng.randint(4, 32), T=_log(rng, 32, 256),
                    H=_log(rng, 64, 512) // 16 * 16, layers=2, V=rng.randint(60, 500))
    return dict(kind="decode", dtype="bf16", B=_log(rng, 1, 256),
                H=_log(rng, 256, 2048) // 64 * 64, layers=rng.randint(1, 4),
                prompt=_log(rng, 64, 1024), V=rng.choice([8000, 16000, 32000]))


# ---- inputs ------------------------------------------------------------------------------
class _Draws:
    """Seeded random tensors on the device."""

    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device=DEVICE).manual_seed(int(seed))

    def normal(self, *shape, scale=1.0):
        return torch.randn(shape, device=DEVICE, generator=self.g).mul_(scale)

    def upstream(self, *shape):
        """A gradient from the layers above: small, and not centred on zero."""
        return self.normal(*shape).add_(1.0).mul_(1e-2)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(shape, device=DEVICE, generator=self.g).mul_(hi - lo).add_(lo)

    def ids(self, hi, *shape):
        return torch.randint(0, hi, shape, device=DEVICE, generator=self.g)


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _module(build, draws: _Draws):
    """``build()`` with trained-looking weights drawn on the device: matrices of unit gain
    (the recurrent ones and the gate's half of it), vectors and gains spread around their
    initial values."""
    with torch.device("meta"):
        module = build()
    module = module.to_empty(device=DEVICE)
    with torch.no_grad():
        for name, p in module.named_parameters():
            leaf = name.rsplit(".", 1)[-1]
            tail = ".".join(name.split(".")[-2:])
            if "embed" in name:
                p.normal_(generator=draws.g).mul_(0.3)
            elif p.dim() == 2:
                gain = (0.5 if tail in ("A.weight", "Ug.weight", "Wg.weight")
                        else 0.1 if "mlp_fc2" in name else 1.0)
                p.normal_(generator=draws.g).mul_(gain / math.sqrt(p.shape[1]))
            else:
                base = BASE.get(tail, BASE.get(leaf, 0.0))
                spread = 0.0 if leaf in FROZEN else 0.1 if p.numel() > 1 else 0.02
                p.normal_(generator=draws.g).mul_(spread).add_(base)
            p.requires_grad_(leaf not in FROZEN)
    return module


def _tapes(draws, B, T, H, dtype):
    """(y, budget, expression, write, novelty, plasticity, energy, saturation) as the core
    scan produces them: signed activations, and rates inside (0, 1)."""
    y = torch.tanh(draws.normal(B, T, H))
    budget = draws.normal(B, T, H, scale=0.7)
    ay = draws.normal(B, T, H, scale=0.5)
    nov = torch.tanh((ay - budget).abs())
    energy = draws.uniform(B, T, H, lo=0.3)
    plast = energy * draws.uniform(B, T, H, lo=0.0, hi=0.8)
    sat = draws.uniform(B, T, H, lo=0.0, hi=0.4)
    return [t.to(dtype) for t in (y, budget, ay, plast * ay, nov, plast, energy, sat)]


def prepare(case, seed):
    kernels.enable("rocm", required=True)
    draws, dt, kind = _Draws(seed), _dtype(case), case["kind"]
    s = {"case": case, "autocast": dt == torch.bfloat16}
    if kind == "scan":
        B, T, D, H = (case[k] for k in "BTDH")
        s["model"] = _module(lambda: dabsn_amd.DABSNCore(D, H), draws)
        s["x"] = draws.normal(B, T, D).to(dt).requires_grad_(True)
        s["up"] = [draws.upstream(B, T, (2 if i == 0 else 1) * H).to(dt)
                   for i in range(7)]
    elif kind == "read":
        B, T, H = (case[k] for k in "BTH")
        s["model"] = _module(lambda: dabsn_amd.DABSNRead(H, case["geometry"]), draws)
        s["tapes"] = [t.requires_grad_(case["train"]) for t in _tapes(draws, B, T, H, dt)]
        if case["train"]:
            s["up"] = draws.upstream(B, T, H)
    elif kind == "long":
        B, T, H = (case[k] for k in "BTH")
        tapes = _tapes(draws, B, T, H, dt)
        s["write"], s["plast"] = (t.requires_grad_(True) for t in (tapes[3], tapes[5]))
        s["logits"] = [(draws.normal(1, scale=0.1) + BASE[n]).requires_grad_(True) for n in (
            "logit_expect_retain", "logit_retention_decay", "logit_retain",
            "logit_retention_strength")]
        s["state"] = [draws.normal(B, H, scale=0.1), draws.normal(B, H, scale=0.1),
                      draws.uniform(B, H)]
        s["up"] = draws.upstream(B, T, H).to(dt)
    elif kind == "delta":
        B, T, H = (case[k] for k in "BTH")
        s["k"] = F.normalize(draws.normal(B, T, H), dim=-1).to(dt).requires_grad_(True)
        s["v"] = draws.normal(B, T, H).to(dt).requires_grad_(True)
        s["beta"] = torch.sigmoid(draws.normal(B, T)).to(dt).requires_grad_(True)
        s["up"] = draws.upstream(B, T, H).to(dt)
    elif kind == "loss":
        N, V, H = (case[k] for k in "NVH")
        s["hidden"] = draws.normal(N, H).to(dt).requires_grad_(True)
        s["weight"] = draws.normal(V, H, scale=1 / math.sqrt(H)).to(dt).requires_grad_(True)
        s["bias"] = draws.normal(V, scale=0.1).to(dt).requires_grad_(True)
        s["targets"] = draws.ids(V, N)
        s["targets"][draws.uniform(N) < 0.1] = -100  # positions without a target
    elif kind == "block":
        B, T, D, H = (case[k] for k in "BTDH")
        s["model"] = _module(lambda: dabsn_amd.DABSNBlock(
            D, D, H, "seq", block_chunk_t=case["chunk"]), draws).train()
        s["x"] = draws.normal(B, T, D).to(dt).requires_grad_(True)
        s["up"] = draws.upstream(B, T, D).to(dt)
    elif kind == "lm":
        H = case["H"]
        s["model"] = _module(lambda: dabsn_amd.DABSNSequenceLM(
            case["V"], H, layers=[(H, H)] * case["layers"]), draws).train()
        s["ids"] = draws.ids(case["V"], case["B"], case["T"])
        s["targets"] = draws.ids(case["V"], case["B"], case["T"])
    else:
        H = case["H"]
        s["model"] = _module(lambda: dabsn_amd.DABSNSequenceLM(
            case["V"], H, layers=[(H, H)] * case["layers"], residual=True, mlp_ratio=4.0),
            draws).to(torch.bfloat16).eval()
        s["memory"] = dabsn_amd.ingest(s["model"], draws.ids(case["V"], case["B"],
                                                             case["prompt"]))
        s["memory"].reserve(case["prompt"] + 1024)
        s["ids"] = draws.ids(case["V"], case["B"], 1)
    return s


# ---- one pass ----------------------------------------------------------------------------
def _gradients(model):
    """The parameters' gradients, those of the one-element gains of a module as one vector."""
    out, gains = {}, {}
    for name, p in model.named_parameters():
        if p.grad is None:
            continue
        if p.numel() == 1:
            parts = name.split(".")
            layer = ".".join(parts[:3]) if parts[0] == "backbone" else ""
            gains.setdefault(layer, []).append(p.grad.reshape(1))
        else:
            out[name] = p.grad
    for layer, g in gains.items():
        out[f"{layer}:gains"] = torch.cat(g)
    return out


def _clear(*tensors, model=None):
    for t in tensors:
        t.grad = None
    if model is not None:
        model.zero_grad(set_to_none=True)


def run(s):
    case = s["case"]
    kind = case["kind"]
    with torch.autocast(DEVICE, torch.bfloat16, enabled=s["autocast"] and kind in (
            "scan", "read", "block")):
        if kind == "scan":
            _clear(s["x"], model=s["model"])
            out = s["model"](s["x"], return_writes=True, return_cocktail=True)
            up = s["up"]
        elif kind == "read":
            if not case["train"]:
                with torch.no_grad():
                    return s["model"](*s["tapes"])
            _clear(*s["tapes"], model=s["model"])
            out = [s["model"](*s["tapes"])]
            up = [s["up"].to(out[0].dtype)]
        elif kind == "block":
            _clear(s["x"], model=s["model"])
            out, up = [s["model"](s["x"])], [s["up"]]
    if kind in ("scan", "read", "block"):
        torch.autograd.backward(out, up)
        inputs = s["tapes"] if kind == "read" else [s["x"]]
        return {"out": list(out), "inputs": [t.grad for t in inputs],
                "params": _gradients(s["model"])}
    if kind == "long":
        _clear(s["write"], s["plast"], *s["logits"])
        out = kernels.long_scan_fused(s["write"], s["plast"], *s["logits"], *s["state"])
        out[0].backward(s["up"])
        return {"out": list(out[:4]), "inputs": [s["write"].grad, s["plast"].grad],
                "logits": torch.cat([t.grad for t in s["logits"]])}
    if kind == "delta":
        _clear(s["k"], s["v"], s["beta"])
        out = kernels.permanent_delta_scan(s["k"], s["v"], s["beta"])
        out.backward(s["up"])
        return {"out": out, "inputs": [s["k"].grad, s["v"].grad, s["beta"].grad]}
    if kind == "loss":
        _clear(s["hidden"], s["weight"], s["bias"])
        loss = dabsn_amd.chunked_linear_cross_entropy(s["hidden"], s["weight"], s["bias"],
                                                      s["targets"])
        loss.backward()
        return {"loss": loss, "inputs": [s["hidden"].grad, s["weight"].grad, s["bias"].grad]}
    if kind == "lm":
        model = s["model"]
        _clear(model=model)
        hidden = model.forward_hidden(s["ids"])
        loss = dabsn_amd.chunked_linear_cross_entropy(hidden, model.readout.weight,
                                                      model.readout.bias, s["targets"])
        loss.backward()
        return {"loss": loss, "hidden": hidden, "params": _gradients(model)}
    logits, s["memory"] = dabsn_amd.forward_with_memory(s["model"], s["ids"], s["memory"],
                                                        extend=True)
    return logits


# ---- what a pass cannot do without -------------------------------------------------------
def work(case):
    kind = case["kind"]
    e = 2 if case["dtype"] == "bf16" else 4
    if kind == "scan":
        B, T, D, H = (case[k] for k in "BTDH")
        rows = B * T
        flops = 6.0 * rows * (2 * D * H + 2 * H * H)
        # x and its gradient, 8 tapes written and as many gradients read, the matrices
        return {"bytes": e * rows * (2 * D + 16 * H) + 8 * (2 * D * H + 2 * H * H),
                "flops": flops}
    if kind == "read":
        B, T, H = (case[k] for k in "BTH")
        pairs = B * T * (T if case["geometry"] == "field" else (T + 1) / 2)
        if case["geometry"] == "hybrid":
            pairs += B * T * T
        proj = 6.0 * B * T * H * H
        flops = 6.0 * H * pairs + proj
        nbytes = e * B * T * H * 8 + 4 * B * T * H + 4 * 3 * H * H
        if case["train"]:
            return {"bytes": 2 * nbytes, "flops": 3 * flops}
        return {"bytes": nbytes, "flops": flops}
    if kind == "long":
        n = case["B"] * case["T"] * case["H"]
        return {"bytes": 6.0 * e * n, "flops": 60.0 * n}
    if kind == "delta":
        B, T, H = (case[k] for k in "BTH")
        return {"bytes": 6.0 * e * B * T * H, "flops": 12.0 * B * T * H * H}
    if kind == "loss":
        N, V, H = (case[k] for k in "NVH")
        return {"bytes": 2.0 * e * (N * H + V * H), "flops": 6.0 * N * V * H}
    if kind == "block":
        B, T, D, H = (case[k] for k in "BTDH")
        rows = B * T
        flops = 6.0 * rows * (2 * D * H + 2 * H * H + 3 * H * H + H * D)
        flops += 18.0 * H * B * T * (T + 1) / 2
        return {"bytes": e * rows * 4 * D + 8.0 * (3 * D * H + 5 * H * H), "flops": flops}
    if kind == "lm":
        B, T, H, L, V = (case[k] for k in ("B", "T", "H", "layers", "V"))
        rows = B * T
        flops = L * (6.0 * rows * 7 * H * H + 18.0 * H * B * T * (T + 1) / 2)
        flops += 6.0 * rows * H * V
        return {"bytes": L * (8.0 * 7 * H * H + 4.0 * rows * H * 2) + 16.0 * V * H,
                "flops": flops}
    B, H, L, N, V = (case[k] for k in ("B", "H", "layers", "prompt", "V"))
    weights = L * (2 + 2 + 3 + 8) * H * H + V * H
    return {"bytes": 2.0 * (L * B * N * H + weights) + 2.0 * B * V,
            "flops": 2.0 * B * weights + L * 6.0 * B * N * H}


# ---- tolerances --------------------------------------------------------------------------
def tolerance(case):
    """About four times the distance to 64 bits of the first kernels, at most 3e-2. The model
    has kinks (the gate's hard limits, the clamped energy, the signs of |expression - budget|
    and |write - expected|): where a value lies on one, two roundings of it take different
    sides, a single gradient element changes altogether, and in a recurrence those before it
    with it. One such element in a short fp32 scan is 3e-3 of a parameter's gradient."""
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if bf16:
        # Recurrent in 16 bits: a rounding of y travels through the later steps.
        rel = {"scan": 3e-2, "block": 3e-2, "read": 2e-2, "decode": 2e-2}.get(kind, 1e-2)
        return {"rel": rel, "max": 0.99}
    rel = {"read": 8e-5, "long": 1e-4, "scan": 1e-2, "lm": 1e-2}.get(kind, 1e-5)
    return {"rel": rel, "max": 0.99 if kind in ("read", "long", "scan", "lm") else 40 * rel}


# ---- 64-bit values -----------------------------------------------------------------------
def _d(t):
    return None if t is None else t.detach().double().requires_grad_(t.requires_grad)


def _core64(x, p):
    """The core recurrence (core.py:171-221) from the zero state: 7 tapes."""
    Wx = F.linear(x, p["W.weight"])
    Wgx = F.linear(x, p["Wg.weight"], p["Wg.bias"])
    fused = torch.cat([p["Ug.weight"], p["A.weight"]])
    alpha = torch.sigmoid(p["logit_alpha"])
    lam, kappa = F.softplus(p["log_lambda"]), F.softplus(p["log_kappa"])
    recover, decay = torch.sigmoid(p["logit_recover"]), torch.sigmoid(p["logit_saturation_decay"])
    sup = torch.sigmoid(p["logit_saturation_suppress"])
    b = torch.zeros_like(Wx[:, 0])
    e, c = torch.ones_like(b), torch.zeros_like(b)
    tapes = [[] for _ in range(7)]
    for t in range(x.shape[1]):
        y = torch.tanh(Wx[:, t] + b)
        rec, ay = F.linear(y, fused).chunk(2, dim=1)
        gate = F.hardsigmoid(Wgx[:, t] + rec)
        nov = torch.tanh((ay - b).abs())
        c = decay * c + (1 - decay) * (nov * (1 - e))
        eff, tb = nov * (1 - sup * c), torch.tanh(b)
        k = (p["k_s"] * gate + p["k_y"] * y + p["k_b"] * tb + p["k_n"] * eff + p["k_bias"]
             + p["k_saturation"] * c)
        r = (p["r_s"] * gate + p["r_y"] * y + p["r_b"] * tb + p["r_n"] * eff + p["r_bias"]
             + p["r_saturation"] * c)
        cost = kappa * torch.exp(0.5 * torch.tanh(k))
        rec_rate = torch.clamp(recover * torch.exp(0.5 * torch.tanh(r)), 0, 1)
        plast = gate * e
        nb = (1 - alpha) * b + p["beta"] + lam * (plast * ay)
        for dst, v in zip(tapes, (torch.cat([y, nb], -1), nov, plast, ay, plast * ay, e, c)):
            dst.append(v)
        b, e = nb, torch.clamp(e + rec_rate * (1 - e) - cost * plast, 0, 1)
    return [torch.stack(v, dim=1) for v in tapes]


def _long64(w, plast, logits, state):
    er, rd, ret, rs = (torch.sigmoid(x) for x in logits)
    L, E, R = state
    out = []
    for wt, pt in zip(w.unbind(1), plast.unbind(1)):
        pe = torch.tanh((wt - E).abs())
        E = er * E + (1 - er) * wt
        R = rd * R + (1 - rd) * (1 - pe)
        eff = ret + (1 - ret) * rs * R
        L = eff * L + (1 - eff) * (pt * pe * wt)
        out.append(L)
    return torch.stack(out, dim=1), (L, E, R)


class _Cast(torch.autograd.Function):
    """A value as the tape dtype holds it; the gradient passes unchanged."""

    @staticmethod
    def forward(ctx, v, dtype):
        return v.to(dtype).to(v.dtype)

    @staticmethod
    def backward(ctx, g):
        return g, None


def _read64(tapes, p, geometry, dtype):
    """The read (read.py:139-438) with dense masks. The means of the tapes, the key bias's
    logarithm and the cocktails are bf16 values where the tapes are, by the read's
    definition: the admitted slots depend on them."""
    y, budget, ay, w, nov, plast, energy, sat = tapes
    B, T, H = ay.shape
    held = (lambda v: v) if dtype == torch.float32 else (lambda v: _Cast.apply(v, dtype))
    me, mc, mn, mp = (held(t.mean(-1)) for t in (energy, sat, nov, plast))
    logp = held(torch.log1p(held(mp * H)))
    g = {k.rsplit(".", 1)[-1]: v for k, v in p.items()}
    kb = g["p_gain"] * logp + g["novelty_gain"] * mn + g["null_bias"]
    adm = (g["adm_p_gain"] * logp + g["adm_novelty_gain"] * mn + g["adm_saturation_gain"] * mc
           + g["adm_energy_gain"] * me + g["adm_bias"])
    stack = torch.stack([me, mc, mn, mp], -1)
    ck = held(stack / held(stack.norm(dim=-1, keepdim=True)).clamp_min(1e-12))
    q, K = F.normalize(ay, dim=-1), F.normalize(w, dim=-1)
    Vn = torch.cat([w[:, 1:], w[:, -1:]], dim=1)
    window = F.softplus(g["admit_window"])
    fixed = adm.detach()
    top = fixed.cummax(1).values if geometry == "seq" else fixed.amax(1, keepdim=True)
    member = (fixed >= top - window).unsqueeze(1)
    qk = (q @ K.transpose(1, 2)) * ((F.softplus(g["log_temp"]) + 1) * math.sqrt(H))
    short = qk + (kb + adm).unsqueeze(1)
    perm = short + g["cocktail_gain"] * (ck @ ck.transpose(1, 2))
    del qk
    pos = torch.arange(T, device=ay.device)

    def weights(scores, allow):
        any_slot = allow.any(-1, keepdim=True)
        scores = scores.masked_fill(~allow, float("-inf")).masked_fill(~any_slot, 0.0)
        return torch.softmax(scores, -1) * any_slot

    def read(causal):
        if causal:
            allow = member & (pos <= pos[:, None])
            induct = member & (pos < pos[:, None])
        else:
            allow = member.expand(B, T, T)
            induct = allow & (pos < T - 1)
        out = (g["short_gain"] * weights(short, allow) + g["pad_gain"] * weights(perm, allow)) @ w
        return out + g["induct_gain"] * (weights(short, induct) @ Vn)

    if geometry == "hybrid":
        gate = torch.sigmoid(g["hybrid_gate"])
        got = (1 - gate) * read(True) + gate * read(False)
    else:
        got = read(geometry == "seq")
    out = F.linear(torch.cat([y, budget, got], -1), p["short_read.out.weight"],
                   p["short_read.out.bias"])
    zero = torch.zeros_like(w[:, 0])
    long, _ = _long64(w, plast, [g[n] for n in (
        "logit_expect_retain", "logit_retention_decay", "logit_retain",
        "logit_retention_strength")], (zero, zero, torch.ones_like(zero)))
    return out + g["long_gain"] * long


def _params64(model, prefix=""):
    return {n[len(prefix):]: _d(v) for n, v in model.named_parameters() if n.startswith(prefix)}


def _exact_gradients(model, p):
    """``_gradients`` of the 64-bit copies ``p``, through the module's own parameters' names."""
    class View:
        @staticmethod
        def named_parameters():
            return [(n, p[n]) for n, _ in model.named_parameters()]
    return _gradients(View)


def _block64(x, p, H, dtype):
    core = {k[5:]: v for k, v in p.items() if k.startswith("core.")}
    read = {k[5:]: v for k, v in p.items() if k.startswith("read.")}
    U, nov, plast, ay, w, e, c = _core64(x, core)
    y, budget = U.split(H, -1)
    out = y + p["read_gain"] * _read64((y, budget, ay, w, nov, plast, e, c), read, "seq", dtype)
    if "state_to_hidden.weight" in p:
        out = F.linear(out, p["state_to_hidden.weight"], p["state_to_hidden.bias"])
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return None  # a 64-bit pass over the whole prompt for every sequence
    if kind in ("block", "scan", "lm") and case["B"] * case["T"] * case["H"] > 1.4e8:
        return None  # minutes of loop steps
    s = prepare(case, seed)
    dt = _dtype(case)
    if kind == "scan":
        x, p = _d(s["x"]), _params64(s["model"])
        out = _core64(x, p)
        torch.autograd.backward(out, [_d(u) for u in s["up"]])
        return {"out": out, "inputs": [x.grad], "params": _exact_gradients(s["model"], p)}
    if kind == "read":
        tapes, p = [_d(t) for t in s["tapes"]], _params64(s["model"])
        if not case["train"]:
            with torch.no_grad():
                return _read64(tapes, p, case["geometry"], dt)
        out = _read64(tapes, p, case["geometry"], dt)
        out.backward(_d(s["up"]))
        return {"out": [out], "inputs": [t.grad for t in tapes],
                "params": _exact_gradients(s["model"], p)}
    if kind == "long":
        w, pl, lg = _d(s["write"]), _d(s["plast"]), [_d(t) for t in s["logits"]]
        out, (L, E, R) = _long64(w, pl, lg, [_d(t) for t in s["state"]])
        out.backward(_d(s["up"]))
        return {"out": [out, L, E, R], "inputs": [w.grad, pl.grad],
                "logits": torch.cat([t.grad for t in lg])}
    if kind == "delta":
        k, v, beta = _d(s["k"]), _d(s["v"]), _d(s["beta"])
        S = k.new_zeros(case["B"], case["H"], case["H"])
        outs = []
        for t in range(case["T"]):
            r = (S @ k[:, t, :, None])[..., 0]
            outs.append(r)
            S = S + (beta[:, t, None] * (v[:, t] - r))[..., None] * k[:, t, None]
        out = torch.stack(outs, 1)
        out.backward(_d(s["up"]))
        return {"out": out, "inputs": [k.grad, v.grad, beta.grad]}
    if kind == "loss":
        h, w, b = _d(s["hidden"]), _d(s["weight"]), _d(s["bias"])
        loss = F.cross_entropy(F.linear(h, w, b), s["targets"])
        loss.backward()
        return {"loss": loss, "inputs": [h.grad, w.grad, b.grad]}
    p = _params64(s["model"])
    if kind == "block":
        x = _d(s["x"])
        out = _block64(x, p, case["H"], dt)
        out.backward(_d(s["up"]))
        return {"out": [out], "inputs": [x.grad], "params": _exact_gradients(s["model"], p)}
    h = F.embedding(s["ids"], p["embed.weight"])
    for i in range(case["layers"]):
        pre = f"backbone.blocks.{i}."
        h = _block64(h, {k[len(pre):]: v for k, v in p.items() if k.startswith(pre)}, case["H"], dt)
    loss = F.cross_entropy(F.linear(h, p["readout.weight"], p["readout.bias"]).flatten(0, 1),
                           s["targets"].flatten())
    loss.backward()
    return {"loss": loss, "hidden": h, "params": _exact_gradients(s["model"], p)}
