"""The work this framework is used for, as cases that can be timed and checked.

Every case goes through the public entry points, with the operands a training
or evaluation program has in hand: the attention-relation KL of one relation
(``attn_kl_align``, with its gradient or without), of all aligned layers
(``relation_kl_loss``), its three stages called one by one, the RoPE pair that
feeds it, the logits KL and the whole loss side of a distillation step.
"""

from __future__ import annotations

import math

import torch

from linearard_amd.attention_KL import attn_kl_align, relation_kl_loss
from linearard_amd.attention_KL.kernel_A import lse_stats
from linearard_amd.attention_KL.kernel_B import kl_forward
from linearard_amd.attention_KL.kernel_C import kl_backward
from linearard_amd.distill import distillation_loss
from linearard_amd.logits_kl import logits_kl
from linearard_amd.rope import rope_pair

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ROPE_BASE = 10000.0
FACTOR = 8.0  # the student's linear RoPE scaling
# float16 trainers scale their loss (the usual start value of a gradient scaler): the losses that are
# means over tokens have gradients below float16's range otherwise
LOSS_SCALE = {"f16": 65536.0, "bf16": 1.0, "f32": 1.0}


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def _align(name, B, H, Hkv, T, D, dtype, mask, causal=True, grad=True):
    """One relation; Hkv == H is the self relation (q is k) of the trainer."""
    return {"name": name, "kind": "align", "B": B, "H": H, "Hkv": Hkv, "T": T, "D": D, "dtype": dtype, "mask": mask,
            "causal": causal, "grad": grad}


def listed():
    return [
        # the smallest call: a smoke test or a debugging run, where only launches and latency count
        _align("align_smallest", 1, 4, 4, 200, 128, "bf16", "none"),
        # one Q/Q relation of a 7B-shaped model at its native context (32 heads, n = 4096)
        _align("align_4k", 1, 32, 32, 4096, 128, "bf16", "none"),
        # the headline workload: 4K -> 32K extension, 32 heads (the largest case)
        _align("align_32k", 1, 32, 32, 32768, 128, "bf16", "none"),
        # grouped queries against fewer keys (q is not k), padded batch, ragged length, 64-wide heads, float16
        _align("align_gqa_padded", 2, 16, 4, 1531, 64, "f16", "i64"),
        # 256-wide heads
        _align("align_d256", 1, 16, 16, 4096, 256, "bf16", "none"),
        # float32 inputs: the benchmark's materialised configuration (32 heads, n = 1024)
        _align("align_f32", 1, 32, 32, 1024, 128, "f32", "none"),
        # evaluation of the loss without a gradient, a batch with padding
        _align("eval_8k", 1, 32, 32, 8192, 128, "bf16", "bool", grad=False),
        # the trainer's relation loss over its aligned layers (Q/Q 32 heads, K/K and V/V 8), two padded
        # sequences, tensors as the attention hook holds them ([B, T, H, D] seen as [B, H, T, D])
        {"name": "layers_2k", "kind": "layers", "L": 4, "B": 2, "H": 32, "Hkv": 8, "T": 2048, "D": 128,
         "dtype": "bf16", "mask": "i64"},
        # the three stages called one by one, at the shape of the utilisation tests (grouped queries on
        # both sides, not causal, float16)
        {"name": "stages_gates", "kind": "stages", "B": 2, "H": 16, "Hkv": 4, "Hkv_t": 2, "T": 2048, "D": 128,
         "Dt": 128, "dtype": "f16", "mask": "none", "causal": False},
        # the RoPE pair of one layer's queries at the native context
        {"name": "rope_4k", "kind": "rope", "B": 1, "H": 32, "T": 4096, "D": 128, "dtype": "bf16"},
        # the logits KL over the kept positions of a 128256-word vocabulary, with its gradient
        {"name": "logits_128k", "kind": "logits", "B": 1, "K": 512, "V": 128256, "dtype": "bf16", "temperature": 1.0,
         "reduction": "mean"},
        # a whole micro-batch: RoPE pairs, the relation loss and the logits KL, both with gradients
        {"name": "step_1k", "kind": "step", "L": 2, "B": 2, "H": 32, "Hkv": 8, "T": 1024, "D": 128, "dtype": "bf16",
         "mask": "i64", "K": 256, "V": 32000, "temperature": 2.0, "lam_L": 0.5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _pairs(T, causal):
    return T * (T + 1) / 2 if causal else float(T) * T


def _fit(c, most):
    """The case with its length shortened until its work is at most `most` flops."""
    while work(c)["flops"] > most:
        c["T"] = max(16, int(c["T"] * 0.8))
    return c


def draw(rng):
    kind = rng.choice(["align"] * 4 + ["f32", "wide", "eval", "layers", "layers", "stages", "stages", "rope", "logits",
                                       "logits", "step"])
    mask = rng.choice(["none", "none", "i64", "bool"])
    half = rng.choice(["bf16", "bf16", "f16"])
    if kind in ("align", "eval"):
        H = rng.choice([1, 2, 4, 8, 8, 16, 32, 32])
        Hkv = rng.choice([H, H, H, max(1, H // 4)])
        c = _align("", rng.choice([1, 1, 2, 3]), H, Hkv, _log_int(rng, 64, 32768), rng.choice([32, 64, 128, 128, 128]), half,
                   mask, rng.random() < 0.85, kind == "align")
        c = _fit(c, 1e13)
    elif kind == "f32":
        c = _fit(_align("", rng.choice([1, 2]), rng.choice([2, 8, 32]), 0, _log_int(rng, 64, 4096),
                        rng.choice([64, 128, 128]), "f32", mask, rng.random() < 0.85), 1e11)
    elif kind == "wide":
        c = _fit(_align("", rng.choice([1, 2]), rng.choice([4, 8, 16]), 0, _log_int(rng, 64, 8192), 256, half, mask), 2e12)
    elif kind == "layers":
        H = rng.choice([8, 16, 32])
        c = _fit({"kind": "layers", "L": rng.choice([1, 2, 3, 4]), "B": rng.choice([1, 2]), "H": H,
                  "Hkv": rng.choice([H, max(1, H // 4)]), "T": _log_int(rng, 128, 8192),
                  "D": rng.choice([64, 128, 128]), "dtype": half, "mask": mask}, 5e12)
    elif kind == "stages":
        H = rng.choice([2, 4, 8, 16])
        c = _fit({"kind": "stages", "B": rng.choice([1, 2, 4]), "H": H, "Hkv": rng.choice([H, max(1, H // 4)]),
                  "Hkv_t": rng.choice([H, max(1, H // 2)]), "T": _log_int(rng, 64, 8192),
                  "D": rng.choice([8, 64, 128, 128, 256]), "Dt": rng.choice([64, 128, 128]), "dtype": half,
                  "mask": mask, "causal": rng.random() < 0.5}, 1e12)
    elif kind == "rope":
        c = {"kind": "rope", "B": rng.choice([1, 2]), "H": rng.choice([8, 32]), "T": _log_int(rng, 64, 32768),
             "D": rng.choice([64, 128, 128]), "dtype": half}
    elif kind == "logits":
        c = {"kind": "logits", "B": rng.choice([1, 2]), "K": _log_int(rng, 8, 512),
             "V": rng.choice([32000, 32768, 50257, 128256, _log_int(rng, 1000, 150000)]),
             "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "temperature": rng.choice([1.0, 1.0, 2.0, 1.5]),
             "reduction": rng.choice(["mean", "mean", "none"])}
    else:
        c = _fit({"kind": "step", "L": rng.choice([1, 2, 3]), "B": rng.choice([1, 2]), "H": 32, "Hkv": 8,
                  "T": _log_int(rng, 256, 4096), "D": 128, "dtype": half, "mask": mask, "K": _log_int(rng, 16, 256),
                  "V": rng.choice([32000, 32768, 128256]), "temperature": rng.choice([1.0, 2.0]), "lam_L": 0.5}, 5e12)
        c["K"] = min(c["K"], c["T"])
    if c["kind"] == "align" and c["Hkv"] == 0:
        c["Hkv"] = c["H"]
    c.pop("name", None)
    return c


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _rotated(x, factor):
    """[B, H, T, D] rotated at positions p / factor (rotate_half layout), in float32."""
    T, D = x.shape[2], x.shape[3]
    inv = 1.0 / ROPE_BASE ** (torch.arange(0, D, 2, device=x.device, dtype=torch.float32) / D)
    ang = torch.arange(T, device=x.device, dtype=torch.float32)[:, None] / factor * inv[None, :]
    c, s = ang.cos(), ang.sin()
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _pair(g, B, H, T, D, dtype, hook=False):
    """(student, teacher) of one projection: the teacher's vectors under its RoPE, the student's (drifted by a
    tenth) under its own.  The spread keeps a token's logit with itself at 8 whatever the head width."""
    std = (64.0 / D) ** 0.25
    s, t = [], []
    for _ in range(H):  # head by head, which bounds the float32 scratch
        x = std * _normal(g, B, 1, T, D)
        s.append(_rotated(x + 0.1 * std * _normal(g, B, 1, T, D), FACTOR).to(dtype))
        t.append(_rotated(x, 1.0).to(dtype))
    s, t = torch.cat(s, 1), torch.cat(t, 1)
    if hook:  # [B, T, H, D] in memory
        s, t = (v.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for v in (s, t))
    return s, t


def _mask(g, kind, B, T):
    """Right padding: sequence b keeps between 60 % and all of its tokens."""
    if kind == "none":
        return None
    keep = (T * (0.6 + 0.4 * torch.rand((B, 1), generator=g, device="cuda"))).long().clamp_min(1)
    m = torch.arange(T, device="cuda")[None, :] < keep
    return m if kind == "bool" else m.to(torch.int64)


def prepare(case, seed):
    g = _gen(seed)
    c, kind = dict(case), case["kind"]
    dt = DTYPES[c["dtype"]]
    st = {"case": c}
    if kind == "align":
        st["mask"] = _mask(g, c["mask"], c["B"], c["T"])
        qs, qt = _pair(g, c["B"], c["H"], c["T"], c["D"], dt)
        qs.requires_grad_(c["grad"])
        ks, kt = qs, qt
        if c["Hkv"] != c["H"]:
            ks, kt = _pair(g, c["B"], c["Hkv"], c["T"], c["D"], dt)
            ks.requires_grad_(c["grad"])
        st.update(qs=qs, ks=ks, qt=qt, kt=kt)
    elif kind == "layers":
        st["mask"] = _mask(g, c["mask"], c["B"], c["T"])
        for n, H in (("q", c["H"]), ("k", c["Hkv"]), ("v", c["Hkv"])):
            pairs = [_pair(g, c["B"], H, c["T"], c["D"], dt, hook=True) for _ in range(c["L"])]
            st[n + "s"] = [p[0].requires_grad_(True) for p in pairs]
            st[n + "t"] = [p[1] for p in pairs]
    elif kind == "stages":
        st["mask"] = _mask(g, c["mask"], c["B"], c["T"])
        st["qs"] = _normal(g, c["B"], c["H"], c["T"], c["D"]).to(dt)
        st["ks"] = _normal(g, c["B"], c["Hkv"], c["T"], c["D"]).to(dt)
        st["qt"] = _normal(g, c["B"], c["H"], c["T"], c["Dt"]).to(dt)
        st["kt"] = _normal(g, c["B"], c["Hkv_t"], c["T"], c["Dt"]).to(dt)
    elif kind == "rope":
        st["x"] = _normal(g, c["B"], c["T"], c["H"], c["D"]).to(dt).permute(0, 2, 1, 3)
    elif kind == "logits":
        t = 3.0 * _normal(g, c["B"], c["K"], c["V"])
        st["s"] = (t + 0.5 * _normal(g, c["B"], c["K"], c["V"])).to(dt).requires_grad_(True)
        st["t"] = t.to(dt)
    else:  # step
        st["mask"] = _mask(g, c["mask"], c["B"], c["T"])
        std = (64.0 / c["D"]) ** 0.25  # as in _pair
        for n, H in (("q", c["H"]), ("k", c["Hkv"]), ("v", c["Hkv"])):  # pre-RoPE projections
            st[n] = [(std * _normal(g, c["B"], c["T"], H, c["D"])).to(dt).permute(0, 2, 1, 3) for _ in range(c["L"])]
        # the value projections differ between the models, the queries and keys through their RoPE
        st["vs"] = [(v + 0.1 * std * _normal(g, *v.shape)).to(dt).requires_grad_(True) for v in st["v"]]
        t = 3.0 * _normal(g, c["B"], c["K"], c["V"])
        st["s"] = (t + 0.5 * _normal(g, c["B"], c["K"], c["V"])).to(dt).requires_grad_(True)
        st["t"] = t.to(dt)
    return st


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "align":
        if not c["grad"]:
            with torch.no_grad():
                return {"loss": attn_kl_align(state["qs"], state["ks"], state["qt"], state["kt"],
                                              attn_mask=state["mask"], causal=c["causal"])}
        loss = attn_kl_align(state["qs"], state["ks"], state["qt"], state["kt"], attn_mask=state["mask"],
                             causal=c["causal"])
        wrt = [state["qs"]] if state["ks"] is state["qs"] else [state["qs"], state["ks"]]
        return {"loss": loss.detach(), "grads": list(torch.autograd.grad(loss, wrt))}
    if kind == "layers":
        loss = relation_kl_loss(state["qs"], state["ks"], state["vs"], state["qt"], state["kt"], state["vt"],
                                attn_mask=state["mask"])
        return {"loss": loss.detach(),
                "grads": list(torch.autograd.grad(loss * LOSS_SCALE[c["dtype"]] if c["dtype"] == "f16" else loss,
                                                  state["qs"] + state["ks"] + state["vs"]))}
    if kind == "stages":
        m, causal = state["mask"], c["causal"]
        lse_s = lse_stats(state["qs"], state["ks"], m, causal)
        lse_t = lse_stats(state["qt"], state["kt"], m, causal)
        loss = kl_forward(state["qs"], state["ks"], lse_s, state["qt"], state["kt"], lse_t, m, causal)
        dq, dk = kl_backward(state["qs"], state["ks"], lse_s, state["qt"], state["kt"], lse_t, m, causal)
        return {"lse_s": lse_s, "lse_t": lse_t, "loss": loss, "dq": dq, "dk": dk}
    if kind == "rope":
        return list(rope_pair(state["x"], ROPE_BASE, {"type": "linear", "factor": FACTOR}))
    if kind == "logits":
        out = logits_kl(state["t"], state["s"], temperature=c["temperature"], reduction=c["reduction"])
        loss = out.mean() if c["reduction"] == "none" else out  # "none": the caller reduces by itself
        if c["dtype"] == "f16":
            loss = loss * LOSS_SCALE["f16"]
        grad, = torch.autograd.grad(loss, [state["s"]])
        return {"kl": out.detach(), "grad": grad}
    scaling = {"type": "linear", "factor": FACTOR}
    q = [rope_pair(x, ROPE_BASE, scaling) for x in state["q"]]
    k = [rope_pair(x, ROPE_BASE, scaling) for x in state["k"]]
    qs, ks = [p[0].requires_grad_(True) for p in q], [p[0].requires_grad_(True) for p in k]
    r = distillation_loss(qs, ks, state["vs"], [p[1] for p in q], [p[1] for p in k], state["v"], state["t"], state["s"],
                          attn_mask=state["mask"], lam_A=1.0, lam_L=c["lam_L"], temperature=c["temperature"])
    loss = r.loss * LOSS_SCALE["f16"] if c["dtype"] == "f16" else r.loss
    grads = torch.autograd.grad(loss, qs + ks + state["vs"] + [state["s"]])
    return {"losses": [x.detach() for x in r], "grads": list(grads)}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    """Bytes: every input read once, every output written once.  Flops: the relations' products in
    linear memory (the maps are not kept between forward and backward): both score products forward
    (4 d per pair), again backward with the two gradient products (8 d); evaluation stops at the forward.
    The other kinds count their elementwise work (a few flops per element)."""
    c, kind = case, case["kind"]
    e = 4 if c["dtype"] == "f32" else 2
    if kind == "align":
        H = c["H"]
        Hkv = c["Hkv"] or H
        elems = c["B"] * c["T"] * c["D"] * (H if Hkv == H else H + Hkv)
        P = c["B"] * H * _pairs(c["T"], c["causal"])
        return {"bytes": elems * e * (3 if c["grad"] else 2), "flops": (12 if c["grad"] else 4) * c["D"] * P}
    if kind in ("layers", "step"):
        heads = c["L"] * (c["H"] + 2 * c["Hkv"])
        elems = c["B"] * c["T"] * c["D"] * heads
        w = {"bytes": elems * e * 3, "flops": 12 * c["D"] * c["B"] * heads * _pairs(c["T"], True)}
        if kind == "step":
            w["bytes"] += 3 * c["B"] * c["K"] * c["V"] * e
            # the pairs: pre-RoPE in, both tensors out
            w["bytes"] += 3 * c["B"] * c["T"] * c["D"] * c["L"] * (c["H"] + c["Hkv"]) * e
        return w
    if kind == "stages":
        B, H, T, D, Dt = c["B"], c["H"], c["T"], c["D"], c["Dt"]
        P = B * H * _pairs(T, c["causal"])
        once = B * T * ((H + c["Hkv"]) * D + (H + c["Hkv_t"]) * Dt) * e
        lse = 2 * B * H * T * 4
        # stage A per side, B and C over both, each a call of its own
        return {"bytes": 3 * once + 3 * lse + B * T * D * (H + c["Hkv"]) * 4,
                "flops": P * (6 * (D + Dt) + 4 * D)}
    if kind == "rope":
        n = c["B"] * c["H"] * c["T"] * c["D"]
        return {"bytes": 3 * n * e, "flops": 6 * n}
    n = c["B"] * c["K"] * c["V"]
    return {"bytes": (2 + 3) * n * e, "flops": 20 * n}  # forward reads both; gradient reads both, writes one


# --------------------------------------------------------------------------
# 64-bit results
# --------------------------------------------------------------------------
def _valid(mask, b, T, device):
    return torch.ones(T, dtype=torch.bool, device=device) if mask is None else mask[b].bool()


def _relation64(qs, ks, qt, kt, mask, causal, grad):
    """(per-row lse_s, lse_t, sum of KL(P_t || P_s), dq, dk) in float64, row block by row block."""
    B, H, T, D = qs.shape
    Hs, Ht = ks.shape[1], kt.shape[1]
    a_s, a_t = 1.0 / math.sqrt(D), 1.0 / math.sqrt(qt.shape[3])
    dev = qs.device
    loss = torch.zeros((), dtype=torch.float64, device=dev)
    lse_s = torch.zeros((B, H, T), dtype=torch.float64, device=dev)
    lse_t = torch.zeros((B, H, T), dtype=torch.float64, device=dev)
    dq = torch.zeros(qs.shape, dtype=torch.float64, device=dev) if grad else None
    dk = torch.zeros(ks.shape, dtype=torch.float64, device=dev) if grad else None
    step = max(64, (1 << 25) // T)
    ninf = float("-inf")
    for b in range(B):
        ok = _valid(mask, b, T, dev)
        for h in range(H):
            Ks, Kt = ks[b, h * Hs // H].double(), kt[b, h * Ht // H].double()
            for i0 in range(0, T, step):
                i1 = min(T, i0 + step)
                n = i1 if causal else T
                v = ok[None, :n] & ok[i0:i1, None]
                if causal:
                    v = v & (torch.arange(n, device=dev)[None, :] <= torch.arange(i0, i1, device=dev)[:, None])
                Q = qs[b, h, i0:i1].double()
                S = (Q @ Ks[:n].T * a_s).masked_fill_(~v, ninf)
                St = (qt[b, h, i0:i1].double() @ Kt[:n].T * a_t).masked_fill_(~v, ninf)
                ls, lt = torch.logsumexp(S, 1), torch.logsumexp(St, 1)
                row = ok[i0:i1]
                lse_s[b, h, i0:i1] = torch.where(row, ls, torch.zeros_like(ls))
                lse_t[b, h, i0:i1] = torch.where(row, lt, torch.zeros_like(lt))
                S = torch.where(v, S - torch.where(row, ls, torch.zeros_like(ls))[:, None], torch.zeros_like(S))
                St = torch.where(v, St - torch.where(row, lt, torch.zeros_like(lt))[:, None], torch.zeros_like(St))
                Pt = St.exp() * v
                loss += (Pt * (St - S)).sum()
                if grad:
                    Dm = S.exp() * v - Pt
                    dq[b, h, i0:i1] = a_s * (Dm @ Ks[:n])
                    dk[b, h * Hs // H, :n] += a_s * (Dm.T @ Q)
    return lse_s, lse_t, loss, dq, dk


def _relations64(xs, xt, ws, mask):
    """sum_r w_r KL_r of self relations and the gradient of each student tensor."""
    losses, grads = [], []
    for x, y, w in zip(xs, xt, ws):
        _, _, l, dq, dk = _relation64(x, x, y, y, mask, True, True)
        losses.append(w * l)
        grads.append(w * (dq + dk))
    return losses, grads


def _denom(c, mask):
    return float(c["B"] * c["T"] if mask is None else max(1, int(mask.sum()))) * c["H"]


def _rope_model(x, factor):
    """The rotation as a model holding x computes it: cos and sin, products and sums in x's dtype."""
    T, D = x.shape[2], x.shape[3]
    inv = 1.0 / ROPE_BASE ** (torch.arange(0, D, 2, dtype=torch.float32) / D)
    inv = (inv / factor).to(x.device)
    ang = torch.arange(T, device=x.device, dtype=torch.float32)[:, None] * inv[None, :]
    cs, sn = (torch.cat((f, f), -1).to(x.dtype) for f in (ang.cos(), ang.sin()))
    return x * cs + torch.cat((-x[..., D // 2:], x[..., :D // 2]), -1) * sn


def _rope64(x, factor):
    T, D = x.shape[2], x.shape[3]
    inv = 1.0 / ROPE_BASE ** (torch.arange(0, D, 2, device=x.device, dtype=torch.float64) / D)
    ang = torch.arange(T, device=x.device, dtype=torch.float64)[:, None] / factor * inv[None, :]
    cs, sn = ang.cos(), ang.sin()
    a, b = x[..., :D // 2].double(), x[..., D // 2:].double()
    return torch.cat((a * cs - b * sn, b * cs + a * sn), -1)


def _logits64(t, s, temperature):
    """Per-position KL and its gradient with respect to s, row block by row block."""
    B, K, V = t.shape
    t2, s2 = t.reshape(-1, V), s.detach().reshape(-1, V)
    kl = torch.zeros(B * K, dtype=torch.float64, device=t.device)
    grad = torch.zeros(B * K, V, dtype=torch.float64, device=t.device)
    for r in range(0, B * K, 64):
        # the tempered logits are tensors of the logits' dtype (the trainer divides them before its softmax)
        lt = torch.log_softmax((t2[r:r + 64] / temperature).double(), 1)
        ls = torch.log_softmax((s2[r:r + 64] / temperature).double(), 1)
        kl[r:r + 64] = (lt.exp() * (lt - ls)).sum(1)
        grad[r:r + 64] = (ls.exp() - lt.exp()) / temperature
    return kl.reshape(B, K), grad.reshape(B, K, V)


def exact(case, seed):
    st = prepare(case, seed)
    c, kind, scale = case, case["kind"], LOSS_SCALE[case["dtype"]]
    with torch.no_grad():
        if kind == "align":
            _, _, loss, dq, dk = _relation64(st["qs"], st["ks"], st["qt"], st["kt"], st["mask"], c["causal"], c["grad"])
            if not c["grad"]:
                return {"loss": loss}
            return {"loss": loss, "grads": [dq + dk] if c["Hkv"] == c["H"] else [dq, dk]}
        if kind == "layers":
            w = [1.0 / (_denom(c, st["mask"]) * c["L"])] * (3 * c["L"])
            losses, grads = _relations64(st["qs"] + st["ks"] + st["vs"], st["qt"] + st["kt"] + st["vt"], w, st["mask"])
            return {"loss": sum(losses), "grads": [x * scale for x in grads]}
        if kind == "stages":
            ls, lt, loss, dq, dk = _relation64(st["qs"], st["ks"], st["qt"], st["kt"], st["mask"], c["causal"], True)
            return {"lse_s": ls, "lse_t": lt, "loss": loss, "dq": dq, "dk": dk}
        if kind == "rope":
            return [_rope64(st["x"], FACTOR), _rope64(st["x"], 1.0)]
        if kind == "logits":
            kl, grad = _logits64(st["t"], st["s"], c["temperature"])
            mean = c["reduction"] == "mean"
            return {"kl": kl.mean() if mean else kl, "grad": grad * scale / (c["B"] * c["K"])}
        # step: the relations of the rotated tensors, rounded as the models hold them
        qs, qt, ks, kt = ([_rope_model(x, f) for x in st[n]]
                          for n, f in (("q", FACTOR), ("q", 1.0), ("k", FACTOR), ("k", 1.0)))
        w = [1.0 / _denom(c, st["mask"])] * (3 * c["L"])
        losses, grads = _relations64(qs + ks + st["vs"], qt + kt + st["v"], w, st["mask"])
        L = c["L"]
        Q, K, V = sum(losses[:L]), sum(losses[L:2 * L]), sum(losses[2 * L:])
        attn = (Q + K + V) / L
        kl, grad = _logits64(st["t"], st["s"], c["temperature"])
        lg = kl.mean()
        return {"losses": [attn + c["lam_L"] * lg, attn, lg, Q, K, V],
                "grads": [x * scale / L for x in grads] + [c["lam_L"] * scale * grad / (c["B"] * c["K"])]}


# --------------------------------------------------------------------------
# tolerance
# --------------------------------------------------------------------------
def tolerance(case):
    """About four times the largest error of any output against exact() seen over the ranges."""
    kind, dt = case["kind"], case["dtype"]
    if dt == "f32":
        return {"rel": 1e-6 if kind == "align" else 1e-4}  # align sums in double; a row's KL is a difference
    if kind == "rope":
        return {"rel": 1e-2 if dt == "bf16" else 2e-3}
    rel = 8e-3 if dt == "bf16" else 3e-3
    if kind in ("layers", "step") or (kind == "align" and case["Hkv"] == case["H"]):
        # self relations: the gradient is a difference of two probability-weighted sums whose largest terms
        # (a token against itself) cancel, so the 16-bit rounding of the probabilities weighs more, the
        # fewer the other tokens
        rel += 0.5 / math.sqrt(case["T"])
    return {"rel": rel}
