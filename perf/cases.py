"""The work this package does for its users, as measurable cases: one pass of each is a call (or a forward and its
backward) through the public functions of ``smel``, at the sizes of the repository's own configurations and around them.

The kinds of case:

  layer    ``smel.moe.moe_forward``: the whole MoE layer (router, int4 and selected bf16 experts with LoRA, shared
           expert, combine), forward only or forward and backward, bf16 or fp32, even or Zipf-skewed routing
  experts  ``smel.moe.routed_experts`` with the routing given, as the Gemma block calls it, forward and backward
  mlp      ``smel.moe.mlp_lora``: the dense gated MLP with LoRA, forward and backward
  ce       ``smel.loss.chunked_ce``: loss and gradient of the rows over a frozen bf16 or int8 head
  norms    every RMSNorm of a block (plain, strided heads, residual add, gated), forward and backward
  quant    ``smel.quant.quantize_int4``: a bank of bf16 experts into the on-disk int4 format

``exact`` restates each in float64 with plain torch. The weights of a quantized bank or head are the values its format
defines for the activations' dtype (dequantized in fp32, rounded once to bf16 where the rows are bf16).

A top-k choice between two experts whose logits agree to the rounding of bf16 is right either way, so the layer's
tokens are drawn with the K-th and the next logit apart by more than two bf16 steps (other tokens are dropped and
replaced before the case starts): every correct implementation then routes alike.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "smel-ft_amd")   # the package of the tree this runs in
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from smel import loss as _loss        # noqa: E402
from smel import lora as _lora        # noqa: E402
from smel import moe as _moe          # noqa: E402
from smel import norm as _norm        # noqa: E402
from smel import quant as _quant      # noqa: E402

DEV = "cuda"
_PROJ = ("A_gate", "B_gate", "A_up", "B_up", "A_down", "B_down")
_DT = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
_EPS = 1e-6

# the two model shapes of the configurations: hidden, experts, expert intermediate, top-k, shared / dense intermediate
_QWEN = {"H": 2048, "E": 256, "I": 512, "K": 8, "Is": 512}
_GEMMA = {"H": 2816, "E": 128, "I": 704, "K": 8, "Is": 2112}


def _layer(T, train, dtype="bf16", zipf=False, n_sel=12, r=16):
    return {"kind": "layer", **_QWEN, "T": T, "train": train, "dtype": dtype, "zipf": zipf, "n_sel": n_sel, "r": r}


def listed():
    return [
        # a short prompt scored without gradients: every launch is small, latency and launches count
        {"name": "layer_eval_23", **_layer(23, False, n_sel=0, r=0)},
        # the evaluation loss of a full packed sequence, every expert frozen int4
        {"name": "layer_eval_4092", **_layer(4092, False, n_sel=0, r=0)},
        # a training step's layer on a short sequence
        {"name": "layer_train_517", **_layer(517, True)},
        # the fine-tuning step itself: forward and backward of the layer over a full packed sequence
        {"name": "layer_train_4092", **_layer(4092, True)},
        # the same with a skewed expert popularity, the popular experts being the trained ones
        {"name": "layer_train_zipf_4096", **_layer(4096, True, zipf=True)},
        # a model kept in float32 (comparisons, gradient checks)
        {"name": "layer_train_f32_1021", **_layer(1021, True, dtype="f32")},
        # the routed experts of a Gemma-style block (GELU, wider hidden size), forward and backward
        {"name": "experts_gemma_4096", "kind": "experts", **_GEMMA, "T": 4096, "n_sel": 12, "r": 16},
        # its dense MLP with LoRA, on one document of a packed batch
        {"name": "mlp_gemma_1531", "kind": "mlp", "H": _GEMMA["H"], "Is": _GEMMA["Is"], "T": 1531, "r": 16,
         "act": "gelu_tanh"},
        # the loss of a full sequence over the bf16 head
        {"name": "ce_4092", "kind": "ce", "N": 4092, "H": 2048, "V": 248320, "int8": False, "softcap": 0.0,
         "dtype": "bf16"},
        # the supervised rows of a short batch over an int8 head with the final-logit softcap
        {"name": "ce_int8_softcap_777", "kind": "ce", "N": 777, "H": 2816, "V": 131072, "int8": True, "softcap": 30.0,
         "dtype": "bf16"},
        # every norm of a block over a full sequence
        {"name": "norms_4092", "kind": "norms", "T": 4092, "H": 2048, "dtype": "bf16"},
        # packing a layer: the gate_up bank of all experts to int4
        {"name": "quant_bank_256", "kind": "quant", "E": 256, "R": 1024, "C": 2048, "group": 64, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "experts", "mlp", "ce", "norms", "quant"])
    if kind == "layer":
        train = rng.random() < 0.7
        if train and rng.random() < 0.25:
            return _layer(_log_int(rng, 64, 1021), True, dtype="f32", r=rng.choice([8, 16, 32]),
                          n_sel=rng.choice([4, 12]))
        if not train:
            return _layer(_log_int(rng, 16, 4092), False, n_sel=0, r=0)
        return _layer(_log_int(rng, 128, 4092), True, zipf=rng.random() < 0.3, n_sel=rng.choice([4, 12, 16]),
                      r=rng.choice([8, 16, 16, 32]))
    if kind == "experts":
        return {"kind": "experts", **_GEMMA, "T": _log_int(rng, 256, 4096), "n_sel": rng.choice([4, 12]),
                "r": rng.choice([8, 16])}
    if kind == "mlp":
        return {"kind": "mlp", "H": rng.choice([2048, 2816]), "Is": rng.choice([512, 1408, 2112]),
                "T": _log_int(rng, 128, 4096), "r": rng.choice([8, 16, 32]), "act": rng.choice(["silu", "gelu_tanh"])}
    if kind == "ce":
        return {"kind": "ce", "N": _log_int(rng, 128, 2048), "H": rng.choice([2048, 2816]),
                "V": rng.randrange(32000, 152000), "int8": rng.random() < 0.4,
                "softcap": rng.choice([0.0, 0.0, 30.0]), "dtype": "bf16"}
    if kind == "norms":
        return {"kind": "norms", "T": _log_int(rng, 64, 4096), "H": rng.choice([2048, 2816, 4096]),
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    return {"kind": "quant", "E": rng.randrange(16, 257), "R": rng.choice([1024, 1408, 2048]),
            "C": rng.choice([512, 704, 2048]), "group": rng.choice([32, 64, 64]), "dtype": "bf16"}


# ---------------------------------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _int4(w, group):
    """{"q", "scale", "zero"} of w [E, R, C] from each group's own range (the format the package reads)."""
    out = {"q": [], "scale": [], "zero": []}
    for part in w.split(32):
        v = part.float().reshape(*part.shape[:-1], -1, group)
        mn, mx = v.amin(-1, keepdim=True), v.amax(-1, keepdim=True)
        s = ((mx - mn) / 15).clamp_min(1e-8).to(torch.bfloat16)
        z = mn.to(torch.bfloat16)
        q = torch.round((v - z.float()) / s.float()).clamp_(0, 15).to(torch.uint8).reshape(part.shape)
        out["q"].append(q[..., 0::2] | (q[..., 1::2] << 4))
        out["scale"].append(s.squeeze(-1))
        out["zero"].append(z.squeeze(-1))
    return {k: torch.cat(v) for k, v in out.items()}


def _lora_factors(g, lead, H, I, r):
    """fp32 factors as training has them: A uniform in +-1/sqrt(in), B moved away from its zero start."""
    def a(n):
        return (torch.rand(*lead, r, n, generator=g, device=DEV) * 2 - 1) / math.sqrt(n)

    def b(n):
        return torch.randn(*lead, n, r, generator=g, device=DEV) * 0.02
    return {"A_gate": a(H), "B_gate": b(I), "A_up": a(H), "B_up": b(I), "A_down": a(I), "B_down": b(H)}


def _bank(g, c):
    gu, dn = _randn(g, c["E"], 2 * c["I"], c["H"], std=0.02), _randn(g, c["E"], c["H"], c["I"], std=0.02)
    return gu, dn


def _layer_inputs(c, seed):
    """Plain tensors of a layer case (also what the float64 restatement reads)."""
    g = _gen(seed)
    T, H, E, K, Is, n_sel = c["T"], c["H"], c["E"], c["K"], c["Is"], c["n_sel"]
    gate = torch.randn(E, H, generator=g, device=DEV) * 0.02
    x = torch.randn(3 * T + 64, H, generator=g, device=DEV)
    perm = torch.randperm(E, generator=torch.Generator().manual_seed(int(seed) + 1))
    if c["zipf"]:   # expert of popularity rank k gets the logit bias -0.54 ln k through a unit mean of x
        rank = torch.empty(E, dtype=torch.long)
        rank[perm] = torch.arange(E)
        bias = (-0.54 * torch.log(rank.double() + 1.0)).float().to(DEV)
        gate = gate - gate.mean(1, keepdim=True) + (bias / H)[:, None]
        x = x + 1.0
    x, gate = x.to(torch.bfloat16), gate.to(torch.bfloat16)
    top = torch.topk(x.double() @ gate.double().t(), K + 1, dim=1).values
    gap = 2.0 ** -6 * torch.maximum(top[:, K - 1].abs(), top[:, K].abs()).clamp_min(2.0 ** -4)
    x = x[torch.argsort((top[:, K - 1] - top[:, K] < gap).to(torch.int8), stable=True)[:T]].contiguous()
    sel = (perm[:n_sel].tolist() if c["zipf"] else list(range(0, E, E // n_sel))[:n_sel]) if n_sel else []
    gu, dn = _bank(g, c)
    d = {"x": x, "gate": gate, "sel": sel, "gu": _int4(gu, 64), "dn": _int4(dn, 64),
         "sel_gu": gu[sel].clone(), "sel_dn": dn[sel].clone(),
         "sh_gate": _randn(g, Is, H, std=0.02), "sh_up": _randn(g, Is, H, std=0.02),
         "sh_down": _randn(g, H, Is, std=0.02), "sh_sg": _randn(g, 1, H, std=0.02)}
    del gu, dn
    r = c["r"]
    d["lora_ex"] = _lora_factors(g, (len(sel),), H, c["I"], r) if r and sel else None
    d["lora_sh"] = _lora_factors(g, (), H, Is, r) if r else None
    d["gy"] = _randn(g, T, H, std=1e-3)
    if c["dtype"] == "f32":
        for k in ("x", "gate", "sel_gu", "sel_dn", "sh_gate", "sh_up", "sh_down", "sh_sg", "gy"):
            d[k] = d[k].float()
    return d


def _experts_inputs(c, seed):
    g = _gen(seed)
    T, H, E, K, n_sel, r = c["T"], c["H"], c["E"], c["K"], c["n_sel"], c["r"]
    x = _randn(g, T, H)
    probs = torch.softmax(torch.randn(T, E, generator=g, device=DEV) * 1.1, -1)
    topv, topi = torch.topk(probs, K, dim=1)
    topv = topv / topv.sum(-1, keepdim=True) * (0.5 + torch.rand(E, generator=g, device=DEV))[topi]
    sel = list(range(0, E, E // n_sel))[:n_sel]
    gu, dn = _bank(g, c)
    d = {"x": x, "topv": topv, "topi": topi, "sel": sel, "gu": _int4(gu, 64), "dn": _int4(dn, 64),
         "sel_gu": gu[sel].clone(), "sel_dn": dn[sel].clone(), "lora_ex": _lora_factors(g, (len(sel),), H, c["I"], r)}
    d["gy"] = _randn(g, T, H, std=1e-3)
    return d


def _mlp_inputs(c, seed):
    g = _gen(seed)
    T, H, Is = c["T"], c["H"], c["Is"]
    return {"x": _randn(g, T, H), "gate_up": _randn(g, 2 * Is, H, std=0.02), "down": _randn(g, H, Is, std=0.02),
            "lora": _lora_factors(g, (), H, Is, c["r"]), "gy": _randn(g, T, H, std=1e-3)}


def _ce_inputs(c, seed):
    g = _gen(seed)
    w = torch.randn(c["V"], c["H"], generator=g, device=DEV) * 0.02
    d = {"h": _randn(g, c["N"], c["H"], dtype=_DT[c["dtype"]]),
         "tgt": torch.randint(0, c["V"], (c["N"],), generator=g, device=DEV)}
    if c["int8"]:
        s = (w.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-12)
        d["w8"] = {"q": torch.round(w / s).clamp_(-127, 127).to(torch.int8), "scale": s.squeeze(-1).to(torch.bfloat16)}
    else:
        d["w"] = w.to(_DT[c["dtype"]])
    return d


_HD, _NQ, _NKV, _VD, _NV = 256, 16, 2, 128, 32   # q / k heads and the gated output heads of a block


def _norms_inputs(c, seed):
    g, dt = _gen(seed), _DT[c["dtype"]]
    T, H = c["T"], c["H"]
    rn = lambda *s, std=1.0: _randn(g, *s, std=std, dtype=dt)
    return {"h": rn(T, H), "a": rn(T, H), "qg": rn(T, _NQ, 2 * _HD), "k": rn(T, _NKV, _HD), "o": rn(T, _NV, _VD),
            "z": rn(T, _NV, _VD), "w_in": rn(H, std=0.1), "w_post": rn(H, std=0.1), "w_q": rn(_HD, std=0.1),
            "w_k": rn(_HD, std=0.1), "w_g": (1 + 0.1 * torch.randn(_VD, generator=g, device=DEV)).to(dt),
            "g_in": rn(T, H), "g_q": rn(T, _NQ, _HD), "g_k": rn(T, _NKV, _HD), "g_s": rn(T, H), "g_y": rn(T, H),
            "g_o": rn(T, _NV, _VD)}


# ------------------------------------------------------------------------------------------------ the package's own


def _module(cls, args, factors):
    m = cls(*args).to(DEV)
    with torch.no_grad():
        for n in _PROJ:
            getattr(m, n).copy_(factors[n])
    return m


def _layer_experts(c, d, act, dtype=torch.bfloat16):
    bank = _moe.Int4Experts(d["gu"], d["dn"], dtype=dtype)
    if not d["sel"]:
        return _moe.LayerExperts(bank, act=act)
    return _moe.LayerExperts(bank, d["sel"], d["sel_gu"], d["sel_dn"], act=act)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "layer":
        d = _layer_inputs(c, seed)
        pre = "mlp.shared_expert"
        W = {"mlp.gate.weight": d["gate"], pre + ".gate_proj.weight": d["sh_gate"], pre + ".up_proj.weight": d["sh_up"],
             pre + ".down_proj.weight": d["sh_down"], pre + "_gate.weight": d["sh_sg"]}
        lora = None
        if c["r"]:
            a = (c["H"], c["I"], c["r"], 2.0 * c["r"])
            lora = _lora.LayerLoRA(
                _module(_lora.ExpertsLoRA, (d["sel"], *a), d["lora_ex"]) if d["lora_ex"] is not None else None,
                _module(_lora.MLPLoRA, (c["H"], c["Is"], c["r"], 2.0 * c["r"]), d["lora_sh"]))
        return {"c": c, "x": d["x"].requires_grad_(c["train"]), "W": W, "lora": lora, "gy": d["gy"],
                "ex": _layer_experts(c, d, "silu", _DT[c["dtype"]])}
    if kind == "experts":
        d = _experts_inputs(c, seed)
        return {"c": c, "x": d["x"].requires_grad_(True), "topv": d["topv"].requires_grad_(True), "topi": d["topi"],
                "ex": _layer_experts(c, d, "gelu_tanh"), "gy": d["gy"],
                "lora": _module(_lora.ExpertsLoRA, (d["sel"], c["H"], c["I"], c["r"], 2.0 * c["r"]), d["lora_ex"])}
    if kind == "mlp":
        d = _mlp_inputs(c, seed)
        Is = c["Is"]
        return {"c": c, "x": d["x"].requires_grad_(True), "gate_up": d["gate_up"], "gate": d["gate_up"][:Is],
                "up": d["gate_up"][Is:], "down": d["down"], "gy": d["gy"],
                "lora": _module(_lora.MLPLoRA, (c["H"], Is, c["r"], 2.0 * c["r"]), d["lora"])}
    if kind == "ce":
        d = _ce_inputs(c, seed)
        head = (_loss.LMHead(int8=d["w8"], softcap=c["softcap"]) if c["int8"] else
                _loss.LMHead(weight=d["w"], softcap=c["softcap"]))
        return {"c": c, "h": d["h"].requires_grad_(True), "tgt": d["tgt"], "head": head}
    if kind == "norms":
        d = _norms_inputs(c, seed)
        for k in ("h", "a", "qg", "k", "o", "z"):
            d[k].requires_grad_(True)
        return {"c": c, **d}
    w = _randn(_gen(seed), c["E"], c["R"], c["C"], std=0.02, dtype=_DT[c["dtype"]])
    return {"c": c, "w": w}


def _clear(*leaves):
    for t in leaves:
        t.grad = None


def run(state):
    s, c = state, state["c"]
    kind = c["kind"]
    if kind == "layer":
        if not c["train"]:
            with torch.no_grad():
                return [_moe.moe_forward(s["x"], s["W"], s["ex"], c["K"], None)]
        params = list(s["lora"].parameters())
        _clear(s["x"], *params)
        y = _moe.moe_forward(s["x"], s["W"], s["ex"], c["K"], s["lora"])
        y.backward(s["gy"])
        return [y.detach(), s["x"].grad] + [p.grad for p in params]
    if kind == "experts":
        params = list(s["lora"].parameters())
        _clear(s["x"], s["topv"], *params)
        y = _moe.routed_experts(s["x"], s["topv"], s["topi"], s["ex"], s["lora"])
        y.backward(s["gy"])
        return [y.detach(), s["x"].grad, s["topv"].grad] + [p.grad for p in params]
    if kind == "mlp":
        params = list(s["lora"].parameters())
        _clear(s["x"], *params)
        y = _moe.mlp_lora(s["x"], s["gate"], s["up"], s["down"], s["lora"], c["act"], s["gate_up"])
        y.backward(s["gy"])
        return [y.detach(), s["x"].grad] + [p.grad for p in params]
    if kind == "ce":
        _clear(s["h"])
        loss = _loss.chunked_ce(s["h"], s["head"], s["tgt"], c["N"])
        loss.backward()
        return [loss.detach(), s["h"].grad]
    if kind == "norms":
        leaves = [s[k] for k in ("h", "a", "qg", "k", "o", "z")]
        _clear(*leaves)
        y_in = _norm.rmsnorm(s["h"], s["w_in"], _EPS, True)
        y_q = _norm.rmsnorm(s["qg"][..., :_HD], s["w_q"], _EPS, True)
        y_k = _norm.rmsnorm(s["k"], s["w_k"], _EPS, True)
        s_, y_ = _norm.add_rmsnorm(s["h"], s["a"], s["w_post"], _EPS, True)
        y_o = _norm.gated_rmsnorm(s["o"], s["z"], s["w_g"], _EPS)
        outs = [y_in, y_q, y_k, s_, y_, y_o]
        grads = torch.autograd.grad(outs, leaves, [s[k] for k in ("g_in", "g_q", "g_k", "g_s", "g_y", "g_o")])
        return [o.detach() for o in outs] + list(grads)
    q = _quant.quantize_int4(s["w"], c["group"])
    return [q["q"], q["scale"], q["zero"]]


# ------------------------------------------------------------------------------------------------ float64


def _deq(d, e, dtype):
    """Expert e of a bank as the values its format defines for rows of ``dtype``, in float64."""
    q = d["q"][e]
    v = torch.stack((q & 15, q >> 4), -1).reshape(q.shape[0], q.shape[1] * 2).float()
    g = v.shape[1] // d["scale"].shape[-1]
    w = v * d["scale"][e].float().repeat_interleave(g, 1) + d["zero"][e].float().repeat_interleave(g, 1)
    return w.to(dtype).double()


def _act64(g, name):
    return torch.nn.functional.silu(g) if name == "silu" else torch.nn.functional.gelu(g, approximate="tanh")


def _mlp64(x, gu, dn, act, f=None, scale=2.0):
    """Gated MLP over rows x, with the LoRA factors f (dict of float64 leaves) on the three projections."""
    h = x @ gu.t()
    I = gu.shape[0] // 2
    g, u = h[:, :I], h[:, I:]
    if f is not None:
        g = g + scale * (x @ f["A_gate"].t()) @ f["B_gate"].t()
        u = u + scale * (x @ f["A_up"].t()) @ f["B_up"].t()
    a = _act64(g, act) * u
    y = a @ dn.t()
    if f is not None:
        y = y + scale * (a @ f["A_down"].t()) @ f["B_down"].t()
    return y


def _leaves64(f):
    return None if f is None else {k: v.double().requires_grad_(True) for k, v in f.items()}


def _routed64(x, topv, topi, d, act, lora, dtype):
    out = torch.zeros_like(x)
    slot = {e: j for j, e in enumerate(d["sel"])}
    for e in range(d["gu"]["q"].shape[0]):
        tok, k = torch.where(topi == e)
        if tok.numel() == 0:
            continue
        if e in slot:
            j = slot[e]
            gu, dn = d["sel_gu"][j].double(), d["sel_dn"][j].double()
            f = {n: lora[n][j] for n in _PROJ} if lora is not None else None
        else:
            gu, dn, f = _deq(d["gu"], e, dtype), _deq(d["dn"], e, dtype), None
        out = out.index_add(0, tok, _mlp64(x[tok], gu, dn, act, f) * topv[tok, k][:, None])
    return out


def _exact_layer(c, seed):
    d, dt = _layer_inputs(c, seed), _DT[c["dtype"]]
    with torch.set_grad_enabled(c["train"]):
        x = d["x"].double().requires_grad_(c["train"])
        lex, lsh = _leaves64(d["lora_ex"]), _leaves64(d["lora_sh"])
        probs = torch.softmax(x @ d["gate"].double().t(), -1)
        topv, topi = torch.topk(probs, c["K"], dim=1)
        topv = topv / topv.sum(-1, keepdim=True)
        y = _routed64(x, topv, topi, d, "silu", lex, dt)
        sh = _mlp64(x, torch.cat((d["sh_gate"], d["sh_up"])).double(), d["sh_down"].double(), "silu", lsh)
        y = y + sh * torch.sigmoid(x @ d["sh_sg"].double().t())
        if not c["train"]:
            return [y]
        y.backward(d["gy"].double())
    grads = [f[n].grad for f in (lex, lsh) if f is not None for n in _PROJ]
    return [y.detach(), x.grad] + grads


def _exact_experts(c, seed):
    d = _experts_inputs(c, seed)
    x, topv, lex = d["x"].double().requires_grad_(True), d["topv"].double().requires_grad_(True), _leaves64(d["lora_ex"])
    y = _routed64(x, topv, d["topi"], d, "gelu_tanh", lex, torch.bfloat16)
    y.backward(d["gy"].double())
    return [y.detach(), x.grad, topv.grad] + [lex[n].grad for n in _PROJ]


def _exact_mlp(c, seed):
    d = _mlp_inputs(c, seed)
    x, f = d["x"].double().requires_grad_(True), _leaves64(d["lora"])
    y = _mlp64(x, d["gate_up"].double(), d["down"].double(), c["act"], f)
    y.backward(d["gy"].double())
    return [y.detach(), x.grad] + [f[n].grad for n in _PROJ]


def _exact_ce(c, seed):
    d, dt = _ce_inputs(c, seed), _DT[c["dtype"]]
    W = d["w"] if not c["int8"] else d["w8"]["q"].to(dt) * d["w8"]["scale"].to(dt)[:, None]
    h, N, cap = d["h"].double(), c["N"], c["softcap"]
    loss, dh = torch.zeros((), dtype=torch.float64, device=DEV), torch.zeros_like(h)
    Wd = W.double()
    for t0 in range(0, N, 1024):
        z = h[t0:t0 + 1024] @ Wd.t()
        t = torch.tanh(z / cap) if cap else None
        zc = t * cap if cap else z
        p = torch.softmax(zc, 1)
        tg = d["tgt"][t0:t0 + 1024, None]
        loss += (torch.logsumexp(zc, 1) - zc.gather(1, tg)[:, 0]).sum()
        p.scatter_add_(1, tg, torch.full(tg.shape, -1.0, dtype=p.dtype, device=DEV))
        if cap:
            p = p * (1 - t * t)
        dh[t0:t0 + 1024] = p @ Wd / N
        del z, zc, p, t
    return [loss / N, dh]


def _rms64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + _EPS) * w


def _exact_norms(c, seed):
    d = _norms_inputs(c, seed)
    v = {k: t.double() for k, t in d.items()}
    leaves = [v[k].requires_grad_(True) for k in ("h", "a", "qg", "k", "o", "z")]
    s = v["h"] + v["a"]
    outs = [_rms64(v["h"], 1 + v["w_in"]), _rms64(v["qg"][..., :_HD], 1 + v["w_q"]), _rms64(v["k"], 1 + v["w_k"]), s,
            _rms64(s, 1 + v["w_post"]), _rms64(v["o"], v["w_g"]) * torch.nn.functional.silu(v["z"])]
    grads = torch.autograd.grad(outs, leaves, [v[k] for k in ("g_in", "g_q", "g_k", "g_s", "g_y", "g_o")])
    return [o.detach() for o in outs] + list(grads)


def exact(case, seed):
    fn = {"layer": _exact_layer, "experts": _exact_experts, "mlp": _exact_mlp, "ce": _exact_ce, "norms": _exact_norms}
    # the quantizer's bytes are defined by fp32 steps and a search between candidates: there is no 64-bit value of them
    return fn[case["kind"]](case, seed) if case["kind"] in fn else None


# ------------------------------------------------------------------------------------------------ work, tolerance


def _mlp_work(rows, H, I, r, train):
    """Products of a gated MLP over ``rows`` rows: forward, and dX; the LoRA factors' products and gradients."""
    f = 2 * rows * 3 * H * I * (2 if train else 1)
    if r:
        f += 2 * rows * r * (3 * (H + I)) * (3 if train else 1)
    return f


def _bank_bytes(n, H, I, group=64):
    return n * 3 * H * I * (0.5 + 4 / group)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("layer", "experts"):
        T, H, I, K, E, r = c["T"], c["H"], c["I"], c["K"], c["E"], c["r"]
        train, esz = c.get("train", True), 4 if c.get("dtype") == "f32" else 2
        used = min(E, T * K)
        n_sel = min(c["n_sel"], used)
        n_lora = T * K * (0.5 if c.get("zipf") else c["n_sel"] / E)   # slots on the trained experts, about
        flops = 2 * T * K * 3 * H * I * (2 if train else 1) + 2 * n_lora * r * 3 * (H + I) * (3 if train else 0)
        nbytes = _bank_bytes(used - n_sel, H, I) + n_sel * 3 * H * I * esz + T * H * esz * 2
        lora = n_sel * r * 3 * (H + I) * 4
        if kind == "layer":
            flops += _mlp_work(T, H, c["Is"], r, train) + 2 * T * H * E * (2 if train else 1)
            nbytes += (3 * H * c["Is"] + E * H) * esz
            lora += r * 3 * (H + c["Is"]) * 4
        else:
            nbytes += T * K * (4 + 8) + (T * K * 4 if train else 0)
        if train:   # the gradients in and out; the weights, read again by the backward, count once
            nbytes += T * H * esz * 2 + 2 * lora
        return {"bytes": int(nbytes), "flops": int(flops)}
    if kind == "mlp":
        T, H, Is, r = c["T"], c["H"], c["Is"], c["r"]
        return {"bytes": 3 * H * Is * 2 + 4 * T * H * 2 + 2 * r * 3 * (H + Is) * 4,
                "flops": _mlp_work(T, H, Is, r, True)}
    if kind == "ce":
        N, H, V = c["N"], c["H"], c["V"]
        return {"bytes": V * H * (1 if c["int8"] else 2) + 2 * N * H * 2 + N * 8, "flops": 4 * N * H * V}
    if kind == "norms":
        T, H = c["T"], c["H"]
        rows = {"in": H * 3, "q": _NQ * _HD * 4, "k": _NKV * _HD * 4, "post": H * 7, "gated": _NV * _VD * 6}
        return {"bytes": 2 * T * sum(rows.values()), "flops": 8 * T * sum(rows.values())}
    n = c["E"] * c["R"] * c["C"]
    return {"bytes": int(n * (2 + 0.5 + 4 / c["group"])), "flops": n * 5 * 8}


def tolerance(case):
    """About four times the largest error of any output against ``exact``: bf16 rounds the activations between the
    products (an output is 3.5e-3 to 5.8e-3 off, its last rounding alone 1.7e-3), fp32 sums over up to 2048 terms."""
    kind, dtype = case["kind"], case.get("dtype", "bf16")
    if kind == "quant":
        return "exact"
    if kind == "layer":
        return {"rel": 6e-6 if dtype == "f32" else 2.3e-2}
    if kind in ("experts", "mlp"):
        return {"rel": 1.7e-2}
    if kind == "ce":
        return {"rel": 7e-3}
    return {"rel": 1.2e-2 if dtype == "bf16" else 1.5e-3}
