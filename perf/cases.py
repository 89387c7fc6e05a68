"""Performance cases: the work that a user of this package has it do, through its public entry points.

Two head layouts occur throughout, both ``ModelArgs`` of this package: ``default`` (1792 wide, 14 heads of 64 + 64,
latent 384, one k_rope per head: the model that is trained) and ``baseline`` (``ModelArgs.mla_baseline``: 2048 wide,
16 heads of 128 + 64, latent 512, one shared k_rope: the dims of the benchmark).  Hidden states are N(0, 1), weights
N(0, 0.02), as in the benchmark.  ``weights`` is ``bf16`` (a module cast to bf16, as it is served) or ``fp32``
(fp32 parameters and residual stream under bf16 autocast, as the training and generation loops run).
"""
import math
from contextlib import nullcontext

import torch

from transformer_amd import MLA, DecodeGraph, ModelArgs, RMSNorm, chunked_linear_cross_entropy

DEV = "cuda"
EPS = 1e-6
CHUNK = 4096  # vocabulary chunk of the loss


def listed():
    return [
        # one user's reply, token by token, a thousand tokens in: the smallest call, where latency counts
        {"name": "decode_one", "kind": "decode", "dims": "baseline", "weights": "bf16", "B": 1, "L": 1000},
        # a serving batch at the context of the decode benchmark
        {"name": "decode_batch", "kind": "decode", "dims": "baseline", "weights": "bf16", "B": 32, "L": 4096},
        # the trained model's own generation: fp32 weights under autocast, one k_rope per head
        {"name": "decode_default", "kind": "decode", "dims": "default", "weights": "fp32", "B": 16, "L": 2500},
        # a prompt read into an empty cache
        {"name": "prompt", "kind": "prompt", "dims": "baseline", "weights": "bf16", "B": 1, "T": 2048},
        # chunks of several prompts continuing a cached prefix (the prefix stays as it is: others continue it too)
        {"name": "chunk", "kind": "chunk", "dims": "baseline", "weights": "bf16", "B": 8, "T": 64, "L": 4000},
        {"name": "chunk_default", "kind": "chunk", "dims": "default", "weights": "fp32", "B": 4, "T": 75, "L": 2500},
        # training, norm and attention of one block, forward and backward: the pretraining shape of the default model
        {"name": "train", "kind": "train", "dims": "default", "weights": "fp32", "B": 6, "T": 2048},
        # the same block fine-tuned on one long document, of any length
        {"name": "train_one", "kind": "train", "dims": "baseline", "weights": "bf16", "B": 1, "T": 3001},
        # attention alone, forward and backward, at the backward benchmark's shape
        {"name": "attention", "kind": "attention", "dims": "baseline", "grad": True, "B": 4, "T": 4096},
        # attention alone, forward, at the long benchmark's shape: no other case has so long a sequence
        {"name": "attention_long", "kind": "attention", "dims": "baseline", "grad": False, "B": 1, "T": 16384},
        # the training loss with its backward
        {"name": "loss", "kind": "loss", "weights": "fp32", "N": 8192, "D": 2048, "V": 32768},
        # the norm inside the down-projections' product, over the pretraining batch
        {"name": "norm_linear", "kind": "norm_linear", "M": 24576, "K": 2048, "N": 2624},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "prompt", "chunk", "train", "attention", "loss", "norm_linear"])
    dims = rng.choice(["baseline", "default"])
    weights = rng.choice(["bf16", "fp32"])
    if kind == "decode":
        B = _log(rng, 1, 64)
        return {"kind": kind, "dims": dims, "weights": weights, "B": B, "L": _log(rng, 100, min(7500, 262144 // B))}
    if kind == "prompt":
        B = _log(rng, 1, 8)
        return {"kind": kind, "dims": dims, "weights": weights, "B": B, "T": _log(rng, 100, 8000 // B)}
    if kind == "chunk":
        B = _log(rng, 1, 16)
        return {"kind": kind, "dims": dims, "weights": weights, "B": B, "T": _log(rng, 8, 256),
                "L": _log(rng, 200, min(7500, 65536 // B))}
    if kind == "train":
        B = _log(rng, 1, 8)
        return {"kind": kind, "dims": dims, "weights": weights, "B": B, "T": _log(rng, 200, min(4000, 12000 // B))}
    if kind == "attention":
        B = _log(rng, 1, 12)
        return {"kind": kind, "dims": dims, "grad": rng.random() < 0.6, "B": B, "T": _log(rng, 200, min(8000, 12000 // B))}
    if kind == "loss":
        return {"kind": kind, "weights": weights, "N": _log(rng, 300, 8000), "D": rng.choice([1024, 1792, 2048]),
                "V": 8 * _log(rng, 1000, 4096)}
    return {"kind": kind, "M": _log(rng, 500, 24000), "K": 32 * _log(rng, 32, 80), "N": 4 * _log(rng, 96, 800)}


# ------------------------------------------------------------------------------------------------ inputs

def _dims(case):
    """(d_model, heads, q_lora, d_latent, nope, v, k_rope heads, RoPE rows)."""
    return (2048, 16, 1024, 512, 128, 128, 1, 16384) if case["dims"] == "baseline" else \
        (1792, 14, 384, 384, 64, 128, 14, 8192)


def _args(case):
    return ModelArgs.mla_baseline() if case["dims"] == "baseline" else ModelArgs()


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _dtype(case):
    return torch.bfloat16 if case["weights"] == "bf16" else torch.float32


def _weights(case, g):
    """One layer's weights by name, in the case's dtype."""
    D, H, ql, dl, dn, dv, hr, _ = _dims(case)
    shapes = {"q_down": (ql, D), "q_up": (H * dn, ql), "qk_rope": ((H + hr) * 64, D), "kv_down": (dl, D),
              "k_up": (H * dn, dl), "v_up": (H * dv, dl), "o_proj": (D, H * dv)}
    return {k: _normal(g, *s, std=0.02, dtype=_dtype(case)) for k, s in shapes.items()}


def _cache(case, g):
    """A cache of L positions as the layer itself leaves it: bf16, latent and rotated keys."""
    _, _, _, dl, _, _, hr, _ = _dims(case)
    return (_normal(g, case["B"], case["L"], dl, dtype=torch.bfloat16),
            _normal(g, case["B"], hr, case["L"], 64, dtype=torch.bfloat16))


def _layer_inputs(case, seed):
    g = _gen(seed)
    T = 1 if case["kind"] == "decode" else case["T"]
    d = {"w": _weights(case, g), "x": _normal(g, case["B"], T, _dims(case)[0], dtype=_dtype(case))}
    if case["kind"] in ("decode", "chunk"):
        d["latent"], d["k_rope"] = _cache(case, g)
    if case["kind"] == "train":
        d["norm"] = 1 + _normal(g, _dims(case)[0], std=0.1)
        d["dy"] = _normal(g, *d["x"].shape, dtype=torch.bfloat16)
    return d


def _attention_inputs(case, seed):
    _, H, _, _, dn, dv, hr, _ = _dims(case)
    B, T, g = case["B"], case["T"], _gen(seed)
    t = [_normal(g, B, T, h, d, dtype=torch.bfloat16) for h, d in ((H, dn), (H, 64), (H, dn), (hr, 64), (H, dv))]
    return t, _normal(g, B, T, H, dv, dtype=torch.bfloat16) if case["grad"] else None


def _loss_inputs(case, seed):
    g = _gen(seed)
    x = _normal(g, 1, case["N"], case["D"], dtype=_dtype(case))
    w = _normal(g, case["V"], case["D"], std=0.02, dtype=_dtype(case))
    return x, w, torch.randint(0, case["V"], (1, case["N"]), generator=g, device=DEV)


def _norm_linear_inputs(case, seed):
    g = _gen(seed)
    return (_normal(g, case["M"], case["K"], dtype=torch.bfloat16),
            _normal(g, case["N"], case["K"], std=0.02, dtype=torch.bfloat16), 1 + _normal(g, case["K"], std=0.1))


def _amp(case):
    return torch.autocast("cuda", torch.bfloat16) if case["weights"] == "fp32" else nullcontext()


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "attention":
        t, s["do"] = _attention_inputs(case, seed)
        s["t"] = [v.requires_grad_(case["grad"]) for v in t]
        s["scale"] = 1 / math.sqrt(_dims(case)[4] + 64)
        return s
    if kind == "loss":
        x, w, s["targets"] = _loss_inputs(case, seed)
        s["x"], s["w"] = x.requires_grad_(True), w.requires_grad_(True)
        return s
    if kind == "norm_linear":
        s["x"], s["w"], s["norm"] = _norm_linear_inputs(case, seed)
        return s
    d = _layer_inputs(case, seed)
    with torch.device(DEV):
        layer = MLA(_args(case))  # fp32 parameters, bf16 RoPE tables
    if case["weights"] == "bf16":
        layer = layer.to(torch.bfloat16)
    layer.load_state_dict({k + ".weight": v for k, v in d["w"].items()})
    s["layer"], s["x"] = layer, d["x"]
    if kind == "train":
        with torch.device(DEV):
            s["norm"] = RMSNorm(_dims(case)[0], eps=EPS)
        s["norm"].load_state_dict({"weight": d["norm"]})
        s["x"].requires_grad_(True)
        s["dy"] = d["dy"]
        s["leaves"] = [s["x"], s["norm"].weight] + [p for _, p in sorted(layer.named_parameters())]
    if kind == "chunk":
        s["cache"] = {"latent": d["latent"], "k_rope": d["k_rope"], "seq_len": case["L"]}
    if kind == "decode":
        with torch.no_grad(), _amp(case):
            s["step"] = DecodeGraph(layer, {"latent": d["latent"], "k_rope": d["k_rope"], "seq_len": case["L"]},
                                    case["L"] + 256)
        s["x"] = s["x"].to(torch.bfloat16)
        n = case["L"] + 1
        s["rows"] = (s["step"].latent[:, :n], s["step"].k_rope[:, :, :n])  # the cache as the step leaves it
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":  # a step at the cache's end
        return (s["step"].step_at(s["x"], case["L"]),) + s["rows"]
    if kind in ("prompt", "chunk"):
        with torch.no_grad(), _amp(case):
            y, cache = s["layer"](s["x"], s.get("cache"), True)
        return y, cache["latent"], cache["k_rope"]
    if kind == "train":
        with _amp(case):
            y, _ = s["layer"](s["norm"](s["x"]))
        return (y,) + torch.autograd.grad(y, s["leaves"], s["dy"])
    if kind == "attention":
        o, lse = torch.ops.mla_mi355x.prefill_fwd(*s["t"], s["scale"], True, 0)
        return (o, lse) if s["do"] is None else (o, lse) + torch.autograd.grad(o, s["t"], s["do"])
    if kind == "loss":
        with _amp(case):
            loss = chunked_linear_cross_entropy(s["x"], s["w"], s["targets"], CHUNK)
        return (loss,) + torch.autograd.grad(loss, [s["x"], s["w"]])
    return torch.ops.mla_mi355x.norm_linear(s["x"], s["w"], s["norm"], EPS)


# ------------------------------------------------------------------------------------------------ what a pass needs

def _size(case):
    return 2 if case["weights"] == "bf16" else 4


def work(case):
    kind = case["kind"]
    if kind == "norm_linear":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 2 * (M * K + N * K + M * N) + 4 * (K + M), "flops": 2 * M * K * N}
    if kind == "loss":
        N, D, V, e = case["N"], case["D"], case["V"], _size(case)
        return {"bytes": 2 * e * (N * D + V * D) + 8 * N, "flops": 6 * N * D * V}  # logits, dx, dw
    D, H, ql, dl, dn, dv, hr, _ = _dims(case)
    B = case["B"]
    if kind == "attention":
        T = case["T"]
        tensors, pairs = B * T * (H * (dn + 64 + dn + dv) + hr * 64), B * H * T * (T + 1) // 2
        flops = 2 * pairs * (dn + 64 + dv)
        if not case["grad"]:
            return {"bytes": 2 * (tensors + B * T * H * dv) + 4 * B * H * T, "flops": flops}
        return {"bytes": 2 * (2 * tensors + 2 * B * T * H * dv) + 4 * B * H * T,
                "flops": flops + 2 * pairs * (3 * (dn + 64) + 2 * dv)}
    down, e = ql + (H + hr) * 64 + dl, _size(case)
    layer = D * down + ql * H * dn + H * dv * D  # products that every new token takes
    weights, up = layer + dl * H * (dn + dv), dl * H * (dn + dv)
    if kind == "decode":
        L = case["L"] + 1
        return {"bytes": 2 * (weights + B * L * (dl + hr * 64) + 2 * B * D),
                "flops": 2 * B * (layer + up + L * H * (2 * dl + 64))}
    T = case["T"]
    L0 = case["L"] if kind == "chunk" else 0
    seen = B * H * (T * L0 + T * (T + 1) // 2)
    row = dl + hr * 64
    if kind == "train":
        flops = 3 * 2 * B * T * weights + 2 * seen * (4 * (dn + 64) + 3 * dv)
        return {"bytes": 2 * e * weights + B * T * D * (2 * e + 4), "flops": flops}
    # keys and values of the whole context, or the absorbed form where that is less
    mix = min(B * (L0 + T) * up + seen * (dn + 64 + dv), B * T * up + seen * (2 * dl + 64))
    return {"bytes": e * weights + 2 * B * row * (L0 + L0 + T) + B * T * D * (e + 2),
            "flops": 2 * (B * T * layer + mix)}


# The relative 2-norm error that bf16 operands and bf16 stored intermediates give, measured against `exact` per kind
# (decode 0.0040, prompt and chunk 0.0038, train 0.0059, attention 0.0025, loss 0.0040, norm_linear 0.0023), times four.
_REL = {"decode": 1.6e-2, "prompt": 1.6e-2, "chunk": 1.6e-2, "train": 2.4e-2, "attention": 1.0e-2, "loss": 1.6e-2,
        "norm_linear": 1.0e-2}


def tolerance(case):
    return {"rel": _REL[case["kind"]]}


# ------------------------------------------------------------------------------------------------ in 64 bits

def _rope64(x, pos):
    """x [B, T, heads, 64] rotated at positions pos + t, with the bf16 tables that are part of the model."""
    f = 1.0 / (10000.0 ** (torch.arange(0, 64, 2).float() / 64))
    a = torch.outer(torch.arange(pos, pos + x.size(1)), f).float()
    c, s = (t.to(torch.bfloat16).double().to(DEV)[None, :, None, :] for t in (a.cos(), a.sin()))
    x1, x2 = x[..., :32], x[..., 32:]
    return torch.cat([x1 * c - x2 * s, x1 * s + x2 * c], -1)


def _attend64(q, k, v, offset):
    """q [T, H, dq], k [L, H, dq], v [L, H, dv]: causal, query t at position offset + t; (o [T, H, dv], lse [H, T])."""
    q, k, v = (t.transpose(0, 1).contiguous() for t in (q, k, v))
    s = torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.size(-1))
    i = torch.arange(q.size(1), device=DEV)[:, None] + offset
    s = s.masked_fill(torch.arange(k.size(1), device=DEV)[None, :] > i, float("-inf"))
    lse = torch.logsumexp(s, -1)
    return torch.bmm(torch.exp(s - lse[..., None]), v).transpose(0, 1), lse


def _layer64(case, w, x, latent=None, k_rope=None):
    """One sequence's layer: (y [T, D], latent [L, dl], k_rope [hr, L, 64]), over a cache where there is one."""
    D, H, ql, dl, dn, dv, hr, _ = _dims(case)
    T, L0 = x.size(0), 0 if latent is None else latent.size(0)
    q = (x @ w["q_down"].t() @ w["q_up"].t()).view(T, H, dn)
    r = _rope64((x @ w["qk_rope"].t()).view(1, T, H + hr, 64), L0)[0]
    lat, kr = x @ w["kv_down"].t(), r[:, H:]
    if L0:
        lat, kr = torch.cat([latent, lat]), torch.cat([k_rope.transpose(0, 1), kr])
    k = torch.cat([(lat @ w["k_up"].t()).view(L0 + T, H, dn), kr.expand(-1, H, -1)], -1)
    o, _ = _attend64(torch.cat([q, r[:, :H]], -1), k, (lat @ w["v_up"].t()).view(L0 + T, H, dv), L0)
    return o.reshape(T, H * dv) @ w["o_proj"].t(), lat, kr.transpose(0, 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "norm_linear":
        x, w, n = (t.double() for t in _norm_linear_inputs(case, seed))
        r = 1 / torch.sqrt((x * x).mean(-1) + EPS)
        return (x * r[:, None] * n) @ w.t(), r
    if kind == "loss":
        x, w, y = _loss_inputs(case, seed)
        x, w, y = x[0].double(), w.double(), y[0]
        p = x @ w.t()
        lse = torch.logsumexp(p, -1)
        loss = (lse - p.gather(1, y[:, None])[:, 0]).mean()
        p = torch.exp(p - lse[:, None])
        p[torch.arange(len(y), device=DEV), y] -= 1
        p /= len(y)
        return loss, (p @ w)[None], p.t().contiguous() @ x
    if kind == "attention":
        t, do = _attention_inputs(case, seed)
        B, T, H, dv = t[4].shape
        o, lse = torch.empty(B, T, H, dv, dtype=torch.float64, device=DEV), torch.empty(B, H, T, dtype=torch.float64, device=DEV)
        grads = [torch.zeros(v.shape, dtype=torch.float64, device=DEV) for v in t]
        for b in range(B):
            for h in range(H):
                hk = h if t[3].size(2) > 1 else 0
                one = [v[b, :, i:i + 1].double().requires_grad_(case["grad"]) for v, i in zip(t, (h, h, h, hk, h))]
                oh, lh = _attend64(torch.cat(one[:2], -1), torch.cat(one[2:4], -1), one[4], 0)
                o[b, :, h], lse[b, h] = oh.detach()[:, 0], lh.detach()[0]
                if case["grad"]:
                    for g, d, i in zip(grads, torch.autograd.grad(oh, one, do[b, :, h:h + 1].double()), (h, h, h, hk, h)):
                        g[b, :, i] += d[:, 0]
        return (o, lse) + (tuple(grads) if case["grad"] else ())
    d = _layer_inputs(case, seed)
    w = {k: v.double() for k, v in d["w"].items()}
    if kind == "train":
        norm = d["norm"].double().requires_grad_(True)
        leaves = [norm] + [v.requires_grad_(True) for _, v in sorted(w.items())]
        ys, dxs, sums = [], [], [torch.zeros_like(v) for v in leaves]
        for b in range(case["B"]):
            x = d["x"][b].double().requires_grad_(True)
            h = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * norm
            y, _, _ = _layer64(case, w, h)
            dx, *g = torch.autograd.grad(y, [x] + leaves, d["dy"][b].double())
            ys.append(y.detach())
            dxs.append(dx)
            for a, v in zip(sums, g):
                a += v
        return (torch.stack(ys), torch.stack(dxs)) + tuple(sums)
    with torch.no_grad():
        x = d["x"].to(torch.bfloat16).double() if kind == "decode" else d["x"].double()
        got = [_layer64(case, w, x[b], *((d["latent"][b].double(), d["k_rope"][b].double()) if "latent" in d else ()))
               for b in range(case["B"])]
        return tuple(torch.stack(v) for v in zip(*got))
