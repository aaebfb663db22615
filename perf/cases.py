"""Performance cases of the library, through its public entry points (include/rabbit_amd.h).

A case is one device call as a decode or prefill loop makes it: the weights are resident, the call is
enqueued on the context's stream and nothing waits for it. The kinds:

    moe      rbt_moe_forward_d: one MoE layer (router, top-k, experts, shared expert, combine)
    latent   rbt_latent_moe_d: K3's MoE layer behind its latent projections
    expert   rbt_apply_single_expert_d: one expert over the tokens that picked it
    matmul   rbt_matmul_qt_d: one quantized projection
    mixers   rbt_gdn_step_d and rbt_gqa_step_d: the two token mixers of one decode token

Shapes are the repository's own workloads (rabbit_amd/workloads.py, bench.py); token counts and
context lengths run from one to the longest prompt a call takes here.
"""
import ctypes as C
import math

import numpy as np
import torch

import rabbit_amd as R
from rabbit_amd import abi
from rabbit_amd.workloads import CONFIGS

# the layers of rabbit_amd/workloads.py
MODELS = {
    "qwen": CONFIGS["c1"],    # hidden 8192, 512 MXFP4 experts of 2048, top-10, gated shared expert
    "k3": CONFIGS["c3"],      # hidden 7168, 384 MXFP4 experts of 2048, top-8, Zipf-skewed routing
    "glm": CONFIGS["c2"],     # hidden 6144, 256 grouped-int4 experts of 2048, top-8
    "latent": CONFIGS["k3l"],  # hidden 7168, 896 MXFP4 experts at 3584 x 3072, top-16
}
# Projections: bench.py's bare-matrix shapes and the latent layer's two projections (columns, rows).
MATRICES = [(7168, 3584), (3584, 7168), (3584, 3072), (4096, 4096), (8192, 2048), (2048, 8192)]
EXPERTS = [(8192, 2048), (7168, 2048), (6144, 2048)]  # (hidden, moe_inter) of the layers above


def listed():
    return [
        # one expert, one token: the reference's apply_single_expert loop at batch 1, the smallest call
        {"name": "expert_token", "kind": "expert", "fmt": "mxfp4", "hidden": 8192, "inter": 2048, "tokens": 1},
        # batch-1 decode of one MXFP4 layer: the benchmark's headline
        {"name": "qwen_decode_1", "kind": "moe", "model": "qwen", "tokens": 1},
        # batched decode, several users at once, skewed routing
        {"name": "k3_decode_8", "kind": "moe", "model": "k3", "tokens": 8},
        # a short prompt (odd length)
        {"name": "qwen_prompt_37", "kind": "moe", "model": "qwen", "tokens": 37},
        # a long prompt (odd length): every expert in use, the largest call
        {"name": "qwen_prompt_1537", "kind": "moe", "model": "qwen", "tokens": 1537},
        # grouped-int4 layer: decode, batched decode, and a prompt (odd length)
        {"name": "glm_decode_1", "kind": "moe", "model": "glm", "tokens": 1},
        {"name": "glm_decode_6", "kind": "moe", "model": "glm", "tokens": 6},
        {"name": "glm_prompt_301", "kind": "moe", "model": "glm", "tokens": 301},
        # the latent layer: decode, and a prompt (odd length)
        {"name": "latent_decode_1", "kind": "latent", "model": "latent", "tokens": 1},
        {"name": "latent_prompt_131", "kind": "latent", "model": "latent", "tokens": 131},
        # a dense projection of a prompt (the latent layer's down projection as the converter writes it)
        {"name": "proj_prompt_77", "kind": "matmul", "fmt": "i4g", "cols": 7168, "rows": 3584, "tokens": 77},
        # the two token mixers of one decode token after a 4K context
        {"name": "mixers_4096", "kind": "mixers", "context": 4096},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "moe", "moe", "latent", "latent", "expert", "matmul", "matmul", "mixers"])
    if kind == "moe":
        model = rng.choice(["qwen", "k3", "glm"])
        return {"kind": kind, "model": model, "tokens": _log_int(rng, 1, 300 if model == "glm" else 1536)}
    if kind == "latent":
        return {"kind": kind, "model": "latent", "tokens": _log_int(rng, 1, 131)}
    if kind == "expert":
        d, i = rng.choice(EXPERTS)
        return {"kind": kind, "fmt": rng.choice(["mxfp4", "i4g"]), "hidden": d, "inter": i, "tokens": _log_int(rng, 1, 256)}
    if kind == "matmul":
        c, r = rng.choice(MATRICES)
        return {"kind": kind, "fmt": rng.choice(["mxfp4", "i4g"]), "cols": c, "rows": r, "tokens": _log_int(rng, 1, 512)}
    return {"kind": "mixers", "context": _log_int(rng, 128, 32768)}


# ---- what a program has in hand -------------------------------------------------------------------
_CTX = None
_FREE = []
_NEXT = 0
DEV = "cuda"


def _context():
    """One context (one stream) for the program; a state holds a layer of it."""
    global _CTX
    if _CTX is None:
        _CTX = R.Context(0)
    return _CTX


class _Layer:
    """A layer number of the context, given back with the state that used it."""

    def __init__(self):
        global _NEXT
        if _FREE:
            self.id = _FREE.pop()
        else:
            self.id = _NEXT
            _NEXT += 1

    def __del__(self):
        _FREE.append(self.id)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _codes(g, *shape):
    """Uniform 4-bit codes, two to a byte."""
    return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=g)


def _normal(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, device=DEV, generator=g) * std + mean


class _Mat:
    """n matrices [rows, cols] of one format in one allocation each for codes and scales."""

    def __init__(self, g, fmt, n, rows, cols, gs=32):
        self.fmt, self.rows, self.cols, self.gs = fmt, rows, cols, gs
        self.data = _codes(g, n, rows, cols // 2)
        if fmt == "mxfp4":
            self.scale = torch.randint(119, 124, (n, rows, cols // 32), dtype=torch.uint8, device=DEV, generator=g)
        else:
            self.scale = torch.rand(n, rows, cols // gs, device=DEV, generator=g) * 0.015 + 0.005

    def qt(self, e):
        if self.fmt == "mxfp4":
            return R.QT.mxfp4(self.data[e], self.scale[e], self.rows, self.cols)
        return R.QT.i4g(self.data[e], self.scale[e], self.rows, self.cols, self.gs)

    def f64(self, e):
        """The dequantized matrix."""
        lut = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0] \
            if self.fmt == "mxfp4" else [float(v - 8) for v in range(16)]
        lut = torch.tensor(lut, dtype=torch.float64, device=DEV)
        b = self.data[e].to(torch.int64)
        w = torch.stack((lut[b & 15], lut[b >> 4]), dim=-1).view(self.rows, -1, self.gs)
        sc = torch.exp2(self.scale[e].double() - 127.0) if self.fmt == "mxfp4" else self.scale[e].double()
        return (w * sc.view(self.rows, -1, 1)).view(self.rows, self.cols)


def _fmt(cfg):
    return "mxfp4" if cfg.kind == R.QT_MXFP4 else "i4g"


def _experts(g, fmt, n, hidden, inter, gs=32):
    return {"gate": _Mat(g, fmt, n, inter, hidden, gs), "up": _Mat(g, fmt, n, inter, hidden, gs),
            "down": _Mat(g, fmt, n, hidden, inter, gs)}


def _slot(m, e, eid=None):
    return R.Slot(e if eid is None else eid, m["down"].qt(e), gate=m["gate"].qt(e), up=m["up"].qt(e))


def _moe(case, seed):
    cfg, S, g = MODELS[case["model"]], case["tokens"], _gen(seed)
    H, E, k = cfg.hidden, cfg.n_experts, cfg.topk
    latent = case["kind"] == "latent"
    d = cfg.extra["moe_hidden"] if latent else H
    s = {"cfg": cfg, "S": S, "layer": _Layer(), "experts": _experts(g, _fmt(cfg), E, d, cfg.inter, cfg.gs),
         "router": _normal(g, E, H, std=cfg.router_std), "x": _normal(g, S, H), "shared": None, "gate": None,
         "bias": None, "lbias": None}
    if cfg.shared:
        s["shared"] = _experts(g, _fmt(cfg), 1, H, cfg.inter, cfg.gs)
    if cfg.gated_shared:
        s["gate"] = _normal(g, H, std=0.02)
    if cfg.family != R.FAMILY_QWEN38 and not cfg.zipf_logit_bias:
        s["bias"] = _normal(g, E, std=0.01)
    if cfg.zipf_logit_bias:
        s["lbias"] = -2.0 * torch.log(torch.randperm(E, device=DEV, generator=g).float() + 1.0)
    s["out"] = torch.empty(S, H, device=DEV)
    s["ids"] = torch.empty(S, k, dtype=torch.int32, device=DEV)
    s["w"] = torch.empty(S, k, device=DEV)
    if latent:
        s["down"] = _Mat(g, "i4g", 1, d, H, cfg.extra["proj_gs"])
        s["up"] = _Mat(g, "i4g", 1, H, d, cfg.extra["proj_gs"])
        s["norm"] = _normal(g, d, std=0.1, mean=1.0)
    return s


def _expert(case, seed):
    S, g = case["tokens"], _gen(seed)
    k = 1 if S == 1 else 8  # a batch's routing: every second token picked this expert
    d, i = case["hidden"], case["inter"]
    s = {"S": S, "k": k, "d": d, "i": i, "m": _experts(g, case["fmt"], 1, d, i), "x": _normal(g, S, d),
         "w": torch.rand(S, k, device=DEV, generator=g), "out": torch.zeros(S, d, device=DEV)}
    ids = torch.randint(1, 256, (S, k), dtype=torch.int32, device=DEV, generator=g)
    ids[::2, k // 2] = 0
    s["ids"] = ids
    return s


def _matmul(case, seed):
    S, g = case["tokens"], _gen(seed)
    return {"S": S, "m": _Mat(g, case["fmt"], 1, case["rows"], case["cols"]), "x": _normal(g, S, case["cols"]),
            "y": torch.empty(S, case["rows"], device=DEV)}


# Qwen 3.8's mixers: 128 V heads over 16 K heads, 128 x 128 state, conv 4; 64 query heads over 4 KV
# heads at head_dim 256, rotary over a quarter of it.
NV, NK, DK, DV, KC = 128, 16, 128, 128, 4
NH, NKV, HD, ROPE, THETA, EPS = 64, 4, 256, 64, 1e7, 1e-6
CONV = 2 * NK * DK + NV * DV


def _mixers(case, seed):
    T, g = case["context"], _gen(seed)
    s = {"T": T, "cap": T + 1}
    s["gdn"] = {"conv_w": _normal(g, CONV, KC, std=0.5), "a_log": _normal(g, NV, std=0.5), "dt": _normal(g, NV, std=0.5),
                "norm": _normal(g, DV, std=0.1, mean=1.0), "conv": _normal(g, CONV, KC - 1),
                "states": _normal(g, NV, DK, DV, std=0.1), "x": _normal(g, CONV), "z": _normal(g, NV * DV),
                "a": _normal(g, NV), "b": _normal(g, NV), "out": torch.empty(NV * DV, device=DEV)}
    s["gqa"] = {"qn": _normal(g, HD, std=0.1), "kn": _normal(g, HD, std=0.1), "kc": _normal(g, T + 1, NKV, HD),
                "vc": _normal(g, T + 1, NKV, HD), "qg": _normal(g, NH, 2, HD), "k": _normal(g, NKV, HD),
                "v": _normal(g, NKV, HD), "out": torch.empty(NH, HD, device=DEV)}
    return s


_MAKE = {"moe": _moe, "latent": _moe, "expert": _expert, "matmul": _matmul, "mixers": _mixers}


def _calls(ctx, case, s):
    """The state's device calls as (entry point, its arguments)."""
    lib, p = ctx.lib, lambda t: t.data_ptr()
    kind = case["kind"]
    if kind == "moe":
        return [(lib.rbt_moe_forward_d, (ctx.h, s["layer"].id, p(s["x"]), s["S"], p(s["out"]), p(s["ids"]), p(s["w"])))]
    if kind == "latent":
        lw = abi.RbtLatentMoeDesc(s["cfg"].extra["moe_hidden"], s["down"].qt(0).c(), s["up"].qt(0).c(), p(s["norm"]), 1e-5,
                                  R.situ(*s["cfg"].extra["situ"]))
        return [(lib.rbt_latent_moe_d, (ctx.h, s["layer"].id, C.byref(lw), p(s["x"]), s["S"], p(s["out"]), p(s["ids"]),
                                        p(s["w"])))]
    if kind == "expert":
        sc = C.pointer(_slot(s["m"], 0).c())
        return [(lib.rbt_apply_single_expert_d, (ctx.h, sc, p(s["ids"]), p(s["w"]), s["S"], s["k"], p(s["x"]), s["d"],
                                                 s["i"], R.ACT_SILU, p(s["out"])))]
    if kind == "matmul":
        q = s["m"].qt(0).c()
        return [(lib.rbt_matmul_qt_d, (ctx.h, p(s["y"]), p(s["x"]), C.byref(q), s["S"]))]
    d, q = s["gdn"], s["gqa"]
    gd = abi.RbtGdnDesc(NV, NK, DK, DV, KC, p(d["conv_w"]), p(d["a_log"]), p(d["dt"]), p(d["norm"]), EPS)
    qd = abi.RbtGqaDesc(NH, NKV, HD, ROPE, THETA, 1.0 / math.sqrt(HD), EPS, p(q["qn"]), p(q["kn"]))
    return [(lib.rbt_gdn_step_d, (ctx.h, C.byref(gd), p(d["conv"]), p(d["states"]), p(d["x"]), p(d["z"]), p(d["a"]),
                                  p(d["b"]), p(d["out"]))),
            (lib.rbt_gqa_step_d, (ctx.h, C.byref(qd), p(q["kc"]), p(q["vc"]), s["cap"], s["T"], p(q["qg"]), p(q["k"]),
                                  p(q["v"]), p(q["out"])))]


def prepare(case, seed):
    ctx = _context()
    s = _MAKE[case["kind"]](case, seed)
    if "layer" in s:
        cfg, layer = s["cfg"], s["layer"].id
        torch.cuda.synchronize()
        for e in range(cfg.n_experts):
            ctx.pool_put(layer, _slot(s["experts"], e))
        ctx.moe_layer_set(layer, cfg.family, cfg.hidden, cfg.inter, cfg.n_experts, cfg.topk, s["router"],
                          shared=_slot(s["shared"], 0, cfg.n_experts) if s["shared"] else None, shared_gate=s["gate"],
                          router_bias=s["bias"], logit_bias=s["lbias"], norm_topk=True, routed_scale=1.0)
    s["calls"] = _calls(ctx, case, s)
    if case["kind"] == "mixers":
        s["outs"] = [s["gdn"]["out"], s["gdn"]["states"], s["gdn"]["conv"], s["gqa"]["out"], s["gqa"]["kc"][s["T"]],
                     s["gqa"]["vc"][s["T"]]]
    elif case["kind"] == "matmul":
        s["outs"] = [s["y"]]
    elif case["kind"] == "expert":
        s["outs"] = [s["out"]]
    else:
        s["outs"] = [s["out"], s["ids"], s["w"]]
    torch.cuda.synchronize()  # the inputs were made on torch's stream
    return s


def run(state):
    ctx = _context()
    for fn, args in state["calls"]:
        rc = fn(*args)
        if rc:
            ctx.check(rc)
    return state["outs"]


# ---- the work ---------------------------------------------------------------------------------------
def _mat_bytes(fmt, rows, cols, gs=32):
    return rows * cols // 2 + rows * (cols // gs) * (1 if fmt == "mxfp4" else 4)


def _unique(case):
    """Experts a call of these tokens picks, on average, under the layer's routing."""
    cfg, S = MODELS[case["model"]], case["tokens"]
    if S == 1:
        return cfg.topk
    r = np.random.default_rng(1)
    logits = r.standard_normal((S, cfg.n_experts)) * cfg.router_std * math.sqrt(cfg.hidden)
    if cfg.zipf_logit_bias:
        logits += 2.0 * np.log(1.0 / (r.permutation(cfg.n_experts) + 1))
    return len(np.unique(np.argpartition(-logits, cfg.topk, axis=1)[:, :cfg.topk]))


def work(case):
    kind = case["kind"]
    if kind in ("moe", "latent"):
        cfg, S = MODELS[case["model"]], case["tokens"]
        H, I, d = cfg.hidden, cfg.inter, cfg.extra.get("moe_hidden", cfg.hidden)
        one = 2 * _mat_bytes(_fmt(cfg), I, d, cfg.gs) + _mat_bytes(_fmt(cfg), d, I, cfg.gs)
        sh = 1 if cfg.shared else 0
        b = (_unique(case) + sh) * one + cfg.n_experts * H * 4 + 2 * S * H * 4 + S * cfg.topk * 8
        f = 2.0 * S * ((cfg.topk + sh) * 3 * I * d + cfg.n_experts * H)
        if kind == "latent":
            b += 2 * _mat_bytes("i4g", d, H, cfg.extra["proj_gs"]) + d * 4
            f += 2.0 * S * 2 * d * H
        return {"bytes": b, "flops": f}
    if kind == "expert":
        S, d, i = case["tokens"], case["hidden"], case["inter"]
        n = (S + 1) // 2
        return {"bytes": 2 * _mat_bytes(case["fmt"], i, d) + _mat_bytes(case["fmt"], d, i) + 3 * n * d * 4,
                "flops": 2.0 * n * 3 * d * i}
    if kind == "matmul":
        S, c, r = case["tokens"], case["cols"], case["rows"]
        return {"bytes": _mat_bytes(case["fmt"], r, c) + S * (c + r) * 4, "flops": 2.0 * S * c * r}
    T = case["context"]
    return {"bytes": 2 * NV * DK * DV * 4 + 2 * CONV * KC * 4 + 3 * NV * DV * 4 + 2 * T * NKV * HD * 4 + 3 * NH * HD * 4,
            "flops": 2.0 * (3 * NV * DK * DV + 2 * T * NH * HD)}


def tolerance(case):
    # prompts of 17 and more tokens round the activations to bf16 on the MXFP4 layers; everything else
    # accumulates fp32 values in fp32
    if case["kind"] == "moe" and case["model"] != "glm" and case["tokens"] > 16:
        return {"rel": 1e-2}
    return {"rel": 4e-6}


# ---- the same in 64 bits ------------------------------------------------------------------------------
def _silu(g):
    return g * torch.sigmoid(g)


def _act(cfg):
    if "situ" not in cfg.extra:
        return lambda g, u: _silu(g) * u
    b, lb = cfg.extra["situ"]
    return lambda g, u: b * torch.tanh(g / b) * torch.sigmoid(g) * (lb * torch.tanh(u / lb))


def _route(s):
    """Expert ids and weights. Selection is by the layer's fp32 logits, a running fp32 sum over the
    columns in order (its near-ties are decided by those bits); the weights are in 64 bits."""
    cfg, x, W = s["cfg"], s["x"], s["router"]
    xt, wt = x.t().contiguous(), W.t().contiguous()
    lg = torch.zeros(x.shape[0], W.shape[0], device=DEV)
    for j in range(W.shape[1]):
        lg += xt[j][:, None] * wt[j][None, :]
    exact = x.double() @ W.double().t()
    if s["lbias"] is not None:
        lg, exact = lg + s["lbias"], exact + s["lbias"].double()
    key = lg
    if cfg.family != R.FAMILY_QWEN38:
        key = torch.sigmoid(lg.double()).float()
        if s["bias"] is not None:
            key = key + s["bias"]
    ids = torch.sort(key, dim=1, descending=True, stable=True)[1][:, :cfg.topk]
    e = torch.gather(exact, 1, ids)
    if cfg.family == R.FAMILY_QWEN38:
        return ids, torch.softmax(e, dim=1)
    p = torch.sigmoid(e)
    return ids, p / (p.sum(1, keepdim=True) + 1e-20)


def _ffn(m, e, x, act):
    return act(x @ m["gate"].f64(e).t(), x @ m["up"].f64(e).t()) @ m["down"].f64(e).t()


def _exact_moe(case, s):
    cfg = s["cfg"]
    ids, w = _route(s)
    x = s["x"].double()
    xe = x @ s["down"].f64(0).t() if case["kind"] == "latent" else x
    out = torch.zeros_like(xe)
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        out[t] += w[t, j][:, None] * _ffn(s["experts"], e, xe[t], _act(cfg))
    if case["kind"] == "latent":
        out = out / torch.sqrt((out * out).mean(1, keepdim=True) + 1e-5) * s["norm"].double()
        out = out @ s["up"].f64(0).t()
    if s["shared"]:
        y = _ffn(s["shared"], 0, x, _act(cfg))
        out += y * torch.sigmoid(x @ s["gate"].double())[:, None] if s["gate"] is not None else y
    return [out, None, w]


def _exact_mixers(s):
    d = {k: v.double() for k, v in s["gdn"].items()}
    hist = torch.cat((d["conv"], d["x"][:, None]), 1)
    c = _silu((d["conv_w"] * hist).sum(1))
    l2 = lambda v: v / torch.clamp(v.norm(dim=1, keepdim=True), min=1e-6)  # noqa: E731
    q = (l2(c[:NK * DK].view(NK, DK)) / math.sqrt(DK)).repeat_interleave(NV // NK, 0)
    k = l2(c[NK * DK:2 * NK * DK].view(NK, DK)).repeat_interleave(NV // NK, 0)
    v = c[2 * NK * DK:].view(NV, DV)
    alpha = torch.exp(-torch.exp(d["a_log"]) * torch.nn.functional.softplus(d["a"] + d["dt"]))
    st = d["states"] * alpha[:, None, None]
    err = v - (k[:, :, None] * st).sum(1)
    st = st + torch.sigmoid(d["b"])[:, None, None] * k[:, :, None] * err[:, None, :]
    o = (q[:, :, None] * st).sum(1)
    o = o / torch.sqrt((o * o).mean(1, keepdim=True) + EPS) * d["norm"]
    o = o.view(-1) * _silu(d["z"])
    a = {n: t.double() for n, t in s["gqa"].items()}
    T = s["T"]
    # rotary angles are fp32 products of the position and an fp32 frequency
    half = ROPE // 2
    inv = torch.tensor(THETA, dtype=torch.float64) ** (-2.0 * torch.arange(half).float() / ROPE).double()
    ang = (torch.tensor(float(T)) * inv.float()).double().to(DEV)

    def rope(h):
        p, r = h[:, :half].clone(), h[:, half:ROPE].clone()
        return torch.cat((p * ang.cos() - r * ang.sin(), r * ang.cos() + p * ang.sin(), h[:, ROPE:]), 1)

    nrm = lambda h, w: h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS) * (1.0 + w)  # noqa: E731
    qh, kh = rope(nrm(a["qg"][:, 0], a["qn"])), rope(nrm(a["k"], a["kn"]))
    kc, vc = a["kc"], a["vc"]
    kc[T], vc[T] = kh, a["v"]
    out = torch.empty(NH, HD, dtype=torch.float64, device=DEV)
    per = NH // NKV
    for h in range(NKV):
        sc = qh[h * per:(h + 1) * per] @ kc[:, h].t() / math.sqrt(HD)
        out[h * per:(h + 1) * per] = torch.softmax(sc, 1) @ vc[:, h].contiguous()
    out = out * torch.sigmoid(a["qg"][:, 1])
    return [o, st, hist[:, 1:].contiguous(), out, kh, a["v"]]


def exact(case, seed):
    s = _MAKE[case["kind"]](case, seed)
    if case["kind"] in ("moe", "latent"):
        return _exact_moe(case, s)
    if case["kind"] == "matmul":
        return [s["x"].double() @ s["m"].f64(0).t()]
    if case["kind"] == "mixers":
        return _exact_mixers(s)
    out = torch.zeros(s["S"], s["d"], dtype=torch.float64, device=DEV)
    t, j = torch.nonzero(s["ids"] == 0, as_tuple=True)
    out[t] = s["w"][t, j].double()[:, None] * _ffn(s["m"], 0, s["x"][t].double(), lambda g, u: _silu(g) * u)
    return [out]
