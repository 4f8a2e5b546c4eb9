"""Workloads of the AttnRes / LR-AttnRes operators, through the drop-in module's public functions.

The cases cover the two read operators (base and LR keys; training, evaluation
and one-token decoding), the cached-logit block schedule of the block decoders
and the value-derived keys, at the sizes of ``bench.py``'s configurations, of
the published whole-model settings, and at ragged ones.

A case is a plain dict.  ``family`` picks the operator; B, T are batch and
tokens, D the model width, N (or S) the depth sources, R / H the LR rank and
heads, Q the read sites of a block phase.
"""

from __future__ import annotations

import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(ROOT, "lr-attnres_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EPS = float(torch.finfo(torch.float32).eps)  # the rms-norms' eps, for every dtype


def _base(name, **kw):
    c = dict(name=name, family="base", B=1, T=1, D=768, N=7, dtype="bf16", train=True, norm=False, counts=False)
    c.update(kw)
    return c


def _lr(name, **kw):
    c = dict(name=name, family="lr", B=1, T=1, D=1024, N=13, R=64, H=4, dtype="bf16", train=True, norm=False,
             counts=False, query="static")
    c.update(kw)
    return c


def listed():
    return [
        # the CPU-sized configuration (fp32, d128, 4 sources): a unit-test sized read, all launch latency
        _base("base_fp32_small", B=2, T=128, D=128, N=4, dtype="fp32", train=False),
        # generation with the block LR model (24 layers, 8 blocks: up to 9 sources): one read site for one new token
        # of 8 sequences, with the count prior and the next sublayer's fused pre-norm; called 48 times a token
        _lr("lr_decode_step", B=8, T=1, D=1024, N=9, R=32, H=1, train=False, norm=True, counts=True),
        # evaluation / prompt processing with the block base model: a read site's forward over whole sequences
        _base("base_eval_norm", B=4, T=2048, D=1024, N=9, train=False, norm=True, counts=True),
        # training the 12-layer d768 model with base keys over block summaries
        _base("base_train_d768", B=8, T=1024, D=768, N=7),
        # training with every sublayer output as a source (24 layers, 48 sublayers): a read site in mid-depth
        _base("base_train_deep", B=4, T=2048, D=1024, N=25),
        # the headline LR read: training, 13 sources, 4 depth heads
        _lr("lr_train_h4", B=8, T=2048, D=1024, N=13, R=64, H=4),
        # training the 12-layer d768 model with LR keys and every sublayer output a source: one depth head (the
        # model's default) and the fused pre-norm, a read site in mid-depth
        _lr("lr_train_h1_d768", B=16, T=1024, D=768, N=13, R=64, H=1, norm=True),
        # fp32 training on ragged sizes (a parity or debugging run)
        _lr("lr_train_fp32_ragged", B=3, T=683, D=640, N=11, R=40, H=5, dtype="fp32"),
        # the widest read: input-dependent gated query, static source keys, 17 sources of 2048
        _lr("lr_train_gated", B=4, T=4096, D=2048, N=17, R=128, H=8, query="gated"),
        # a block of the published block LR decoder (24 layers, 4 blocks): phase 1 for its 12 sites, 11 sublayers
        # grown and read, the completed block source and its logits for the next block's sites
        dict(name="lr_block", family="lr_block", B=8, T=2048, D=1024, S=4, Q=12, R=32, dtype="bf16"),
        # a block of the block base decoder (12 layers, 6 blocks): phase 1 from the block's query bank, then each
        # later site's merge of the live partial block with the fused pre-norm
        dict(name="base_block", family="base_block", B=16, T=1024, D=768, S=6, Q=4, dtype="bf16"),
        # value-derived LR keys of the widest read's sources, and their gradients
        dict(name="value_keys", family="value_keys", B=4, T=4096, D=2048, N=17, R=128, dtype="bf16"),
    ]


def draw(rng):
    """One more case of the same ranges: 1 to 16384 tokens, widths 128 to 2048, 2 to 49 sources."""
    family = rng.choice(["base"] * 4 + ["lr"] * 4 + ["lr_block", "base_block", "value_keys"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "bf16", "bf16", "bf16", "fp16", "fp32"])
    tokens = math.exp(rng.uniform(0.0, math.log(16384.0)))
    B = rng.choice([b for b in (1, 2, 3, 4, 8, 16) if b <= max(1.0, tokens)])
    T = max(1, round(tokens / B))
    if family in ("base", "lr"):
        D = rng.choice([128, 256, 320, 512, 640, 768, 768, 1024, 1024, 1536, 2048, 8 * rng.randint(16, 256)])
        N = round(math.exp(rng.uniform(math.log(2.0), math.log(49.0))))
        train = tokens > 64 and rng.random() < 0.75
        c = dict(family=family, B=B, T=T, D=D, N=N, dtype=dtype, train=train, norm=False, counts=rng.random() < 0.5)
        if family == "base":
            c["norm"] = rng.random() < 0.4
        else:
            c["H"] = rng.choice([h for h in (1, 1, 1, 2, 4, 5, 8, 12) if D % h == 0 and D // h >= 64])
            c["R"] = c["H"] * rng.choice([r for r in (8, 16, 32, 64, 128) if r * c["H"] <= 128])
            c["norm"] = c["H"] == 1 and rng.random() < 0.5
            c["query"] = rng.choice(["static", "static", "static", "token", "gated"])
    elif family == "lr_block":
        c = dict(family=family, B=B, T=T, D=rng.choice([256, 512, 768, 1024, 1024]), S=rng.randint(2, 8),
                 Q=rng.randint(2, 12), R=rng.choice([16, 32, 48, 64, 128]), dtype=rng.choice(["bf16", "bf16", "fp16"]))
    elif family == "base_block":
        c = dict(family=family, B=B, T=T, D=rng.choice([256, 512, 640, 768, 1024]), S=rng.randint(2, 9),
                 Q=rng.randint(2, 12), dtype=rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"]))
    else:
        c = dict(family=family, B=B, T=T, D=rng.choice([256, 512, 768, 1024, 1536, 2048]), N=rng.randint(1, 17),
                 R=rng.choice([32, 64, 128]), dtype="bf16")
    while work(c)["bytes"] > 1.2e9 and c["T"] > 1:
        c["T"] = (c["T"] + 1) // 2
    return c


# ------------------------------------------------------------------ inputs

def _biases(n):
    """The count prior of a block model's sources, log(count): the embedding, whole blocks, a part of one."""
    return [0.0] + [math.log(2.0 + (5 * s) % 7) for s in range(1, n)]


def prepare(case, seed):
    dev = torch.device("cuda")
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    B, T, D = case["B"], case["T"], case["D"]
    family = case["family"]
    st = {"case": case}

    def rn(*shape, std=1.0, dtype=dt):
        return (torch.randn(shape, generator=gen, device=dev) * std).to(dtype)

    if family in ("base", "lr"):
        N, train = case["N"], case["train"]
        # hidden states have unit variance: the embedding, then sublayer outputs or block summaries
        st["values"] = [rn(B, T, D) for _ in range(N)]
        st["bias"] = _biases(N) if case["counts"] else None
        wrt = list(st["values"])
        if family == "base":
            st["query"] = rn(D, std=0.02)
        else:
            R, H = case["R"], case["H"]
            st["keys"] = [rn(B, T, R) for _ in range(N)]
            st["query"] = rn(H, R // H, std=0.5)
            st["scale"] = 1.0 / math.sqrt(R // H)
            wrt += st["keys"]
            if case["query"] == "token":
                st["query"] = rn(B, T, H, R // H, std=0.5)
            elif case["query"] == "gated":
                st["query_dyn"] = rn(B, T, R, std=0.5)
                st["gate"] = rn(B, T, H)
                st["static_keys"] = rn(N, R, std=0.02)
                wrt += [st["query_dyn"], st["gate"], st["static_keys"]]
        wrt.append(st["query"])
        if train:
            st["grad"] = rn(B, T, D)
    elif family == "lr_block":
        S, Q, R = case["S"], case["Q"], case["R"]
        st["values"] = [rn(B, T, D) for _ in range(S)]
        st["logits"] = [rn(Q, B, T, dtype=torch.float32) for _ in range(S)]
        st["projected"] = [rn(B, T, D + R) for _ in range(Q)]  # the sublayers' fused [out | key] projections
        st["bank"] = rn(2 * Q, R, std=0.5)                     # this block's and the next one's site queries
        st["scale"] = 1.0 / math.sqrt(R)
        wrt = st["values"] + st["logits"] + st["projected"] + [st["bank"]]
        st["grad"] = ([rn(B, T, D) for _ in range(Q)] + [rn(B, T, D)] + [rn(Q, B, T, dtype=torch.float32)])
        train = True
    elif family == "base_block":
        S, Q = case["S"], case["Q"]
        st["values"] = [rn(B, T, D) for _ in range(S)]
        st["queries"] = [rn(D, std=0.02) for _ in range(Q)]
        st["partials"] = [rn(B, T, D, std=math.sqrt(q)) for q in range(1, Q)]  # sums of q unit-variance outputs
        wrt = st["values"] + st["queries"] + st["partials"]
        st["grad"] = [rn(B, T, D) for _ in range(Q)]
        train = True
    else:
        N, R = case["N"], case["R"]
        st["values"] = [rn(B, T, D) for _ in range(N)]
        st["weight"] = rn(R, D, std=0.02)
        wrt = st["values"] + [st["weight"]]
        st["grad"] = [rn(B, T, R) for _ in range(N)]
        train = True
    if train:
        for t in wrt:
            t.requires_grad_(True)
        st["wrt"] = wrt
    return st


# ------------------------------------------------------------------ one pass

def _forward(ops, st):
    c = st["case"]
    family = c["family"]
    if family == "base":
        return [ops.attention_residual_read(st["values"], st["query"], True, normalize_output=c["norm"],
                                            source_logit_biases=st["bias"])]
    if family == "lr":
        if c["query"] == "gated":
            return [ops.lrid_attention_residual_read_gated(
                st["values"], st["keys"], st["query"], st["query_dyn"], st["gate"], c["H"], st["scale"], True,
                gate_activation="sigmoid", normalize_output=c["norm"], source_logit_biases=st["bias"],
                static_keys=st["static_keys"])]
        return [ops.lrid_attention_residual_read(st["values"], st["keys"], st["query"], c["H"], st["scale"], True,
                                                 normalize_output=c["norm"], source_logit_biases=st["bias"])]
    if family == "lr_block":
        D, R, Q = c["D"], c["R"], c["Q"]
        inter, lse = ops.lrid_block_phase1(st["values"], st["logits"])
        reads = [inter[0]]
        value = key = None
        for q in range(1, Q):
            value, key, h = ops.lrid_block_accumulate_read(
                st["projected"][q - 1], value, key, st["bank"], inter[q], lse[q], D, R, st["scale"], lerp=True,
                normalize_output=True, logit_bias=math.log(q), partial_scale=1.0 / q, query_row=q)
            reads.append(h)
        value, key = ops.lrid_block_accumulate(st["projected"][Q - 1], value, key, D, R, complete=True,
                                               partial_scale=1.0 / Q)
        (nxt,) = ops.lrid_site_logits(key, st["bank"], Q, [Q], st["scale"], math.log(Q))
        return [*reads, value, nxt]
    if family == "base_block":
        bank = torch.stack(st["queries"])
        inter, lse = ops.attention_residual_phase1(st["values"], bank, True)
        inter, lse = inter.unbind(0), lse.unbind(0)
        reads = [inter[0]]
        for q in range(1, c["Q"]):
            reads.append(ops.attention_residual_phase2(
                st["partials"][q - 1], st["queries"][q], inter[q], lse[q], True, normalize_output=True,
                logit_bias=math.log(q), partial_scale=1.0 / q))
        return reads
    return ops.lrid_value_key_projection(st["values"], st["weight"])


def run(state):
    import attnres_ops as ops

    if "wrt" not in state:
        with torch.no_grad():
            return _forward(ops, state)[0]
    outs = _forward(ops, state)
    g = state["grad"]
    grads = torch.autograd.grad(outs, state["wrt"], g if isinstance(g, list) else [g])
    return [*[o.detach() for o in outs], *grads]


# ------------------------------------------------------------------ the same in 64 bits

def _rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _mix(logits, values, H):
    """softmax over a list of [..., H] logits, mixed over [..., D] values per head."""
    m = torch.stack(logits).max(0).values.detach()
    e = [torch.exp(l - m) for l in logits]
    z = sum(e[1:], e[0])
    out = 0.0
    for x, v in zip(e, values):
        out = out + (x / z).unsqueeze(-1) * v.unflatten(-1, (H, -1))
    return out.flatten(-2), (z.log() + m)


def _exact_forward(c, st):
    family = c["family"]
    D = c["D"]
    if family == "base":
        bias = st["bias"] or [0.0] * c["N"]
        logits = [(_rms(v) * st["query"]).sum(-1, keepdim=True) + b for v, b in zip(st["values"], bias)]
        out, _ = _mix(logits, st["values"], 1)
        return [_rms(out) if c["norm"] else out]
    if family == "lr":
        H, N = c["H"], c["N"]
        bias = st["bias"] or [0.0] * N
        q = st["query"]
        if c["query"] == "gated":
            q = q + torch.sigmoid(st["gate"]).unsqueeze(-1) * st["query_dyn"].unflatten(-1, (H, -1))
        logits = []
        for s in range(N):
            k = st["keys"][s] + st["static_keys"][s] if c["query"] == "gated" else st["keys"][s]
            logits.append((_rms(k.unflatten(-1, (H, -1))) * q).sum(-1) * st["scale"] + bias[s])
        out, _ = _mix(logits, st["values"], H)
        return [_rms(out) if c["norm"] else out]
    if family == "lr_block":
        R, Q = c["R"], c["Q"]
        value = key = 0.0
        reads = []
        for q in range(Q):
            inter, lse = _mix([lg[q].unsqueeze(-1) for lg in st["logits"]], st["values"], 1)
            if q == 0:
                reads.append(inter)
            else:
                value = value + st["projected"][q - 1][..., :D]
                key = key + _rms(st["projected"][q - 1][..., D:])
                logit = (_rms(key) * st["bank"][q]).sum(-1, keepdim=True) * st["scale"] + math.log(q)
                reads.append(_rms(inter + torch.sigmoid(logit - lse) * (value / q - inter)))
        value = (value + st["projected"][Q - 1][..., :D]) / Q
        key = key + _rms(st["projected"][Q - 1][..., D:])
        nxt = (_rms(key) @ st["bank"][Q:].t()).movedim(-1, 0) * st["scale"] + math.log(Q)
        return [*reads, value, nxt]
    if family == "base_block":
        khat = [_rms(v) for v in st["values"]]
        reads = []
        for q in range(c["Q"]):
            inter, lse = _mix([(k * st["queries"][q]).sum(-1, keepdim=True) for k in khat], st["values"], 1)
            if q == 0:
                reads.append(inter)
            else:
                v = st["partials"][q - 1] / q
                logit = (_rms(v) * st["queries"][q]).sum(-1, keepdim=True) + math.log(q)
                reads.append(_rms(inter + torch.sigmoid(logit - lse) * (v - inter)))
        return reads
    return [_rms(v) @ st["weight"].t() for v in st["values"]]


def exact(case, seed):
    """What ``run`` returns for these inputs, in 64 bits, in plain torch."""
    st = prepare(case, seed)
    train = "wrt" in st
    seen = {}

    def up(x):
        if isinstance(x, torch.Tensor):
            if id(x) not in seen:
                seen[id(x)] = x.detach().double().requires_grad_(x.requires_grad)
            return seen[id(x)]
        return [up(t) for t in x] if isinstance(x, list) else x

    d = {k: up(v) for k, v in st.items() if k != "case"}
    if not train:
        with torch.no_grad():
            return _exact_forward(case, d)[0]
    outs = _exact_forward(case, d)
    g = d["grad"]
    grads = torch.autograd.grad(outs, d["wrt"], g if isinstance(g, list) else [g])
    return [*[o.detach() for o in outs], *grads]


# ------------------------------------------------------------------ what a pass needs, and how exact it is

def work(case):
    """Bytes (each input read once, each output written once; what is saved for the backward counts as neither)
    and operations of one pass."""
    c = case
    s = 4 if c["dtype"] == "fp32" else 2
    n, D = c["B"] * c["T"], c["D"]
    family = c["family"]
    if family in ("base", "lr"):
        N = c["N"]
        R, H = (c["R"], c["H"]) if family == "lr" else (0, 1)
        row = N * (D + R)
        dyn = R if family == "lr" and c["query"] != "static" else 0
        dyn += H if family == "lr" and c["query"] == "gated" else 0
        keyw = R if family == "lr" else D
        by = n * (row + D + dyn) * s
        fl = n * N * (2 * D + 4 * keyw)
        if c["train"]:
            by += n * (D + row + row + 2 * dyn) * s  # the backward: gradient in, sources again, their gradients out
            fl += n * N * (3 * D + 8 * keyw)
        return {"bytes": by, "flops": fl}
    if family == "lr_block":
        S, Q, R = c["S"], c["Q"], c["R"]
        W = D + R
        fwd = S * D * s + S * Q * 4 + Q * W * s + Q * D * s + D * s + Q * 4
        bwd = (Q + 1) * D * s + Q * 4 + S * D * s + S * Q * 4 + Q * W * s + S * D * s + S * Q * 4 + Q * W * s
        fl = n * (Q * S * D * 6 + Q * D * 20 + Q * R * 20)
        return {"bytes": n * (fwd + bwd), "flops": fl}
    if family == "base_block":
        S, Q = c["S"], c["Q"]
        ins, outs = S + Q - 1, Q
        return {"bytes": n * D * s * (ins + outs + outs + ins + ins), "flops": n * D * (Q * S * 12 + Q * 24)}
    N, R = c["N"], c["R"]
    return {"bytes": n * N * (D + R + D + R + D) * s, "flops": 6 * n * N * D * R}


def tolerance(case):
    """About four times what the operators show against 64 bits (bf16 has 8 bits of significand, fp16 11)."""
    return {"bf16": {"rel": 2e-2}, "fp16": {"rel": 2.5e-3}, "fp32": {"rel": 1e-5}}[case["dtype"]]
