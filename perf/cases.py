"""Performance cases of the library: what a program that uses it has it do, through the public entry
points of the Python package (one call of the C ABI each).

A whole model's calls are one decode step (forward_pass at a position, which also returns its logits)
and one batched prefill of a prompt (at position 0 or after earlier turns), each on weights uploaded
tensor by tensor as a loader does. Beside them are the calls a host makes itself around or instead of
the model: the sampler over a vocabulary of logits, the attention over a long KV view, and the matrix
product over GGUF blocks or f16 rows. The shapes are the repository's: the stories260K-size model,
TinyLlama 1.1B and Llama-3 8B, at full depth.
"""
import gc
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "runeforgeai-project-aesir_amd"))
import aesir_hip as A  # noqa: E402

MODELS = {
    "tiny": dict(dim=64, n_layers=5, n_heads=8, n_kv_heads=4, ffn=172, vocab=512, theta=10000.0),
    "tinyllama": dict(dim=2048, n_layers=22, n_heads=32, n_kv_heads=4, ffn=5632, vocab=32000, theta=10000.0),
    "llama3": dict(dim=4096, n_layers=32, n_heads=32, n_kv_heads=8, ffn=14336, vocab=128256, theta=500000.0),
}
EPS = 1e-5
STD = 0.02
TYPES = {"f16": 1, "q4_0": 2, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest model's decode step: launches and the host round trip
        dict(name="tiny_decode_f16", kind="decode", model="tiny", type="f16", pos=80),
        # a small chat model generating, f16 and 8-bit
        dict(name="tinyllama_decode_f16", kind="decode", model="tinyllama", type="f16", pos=383),
        dict(name="tinyllama_decode_q8_0", kind="decode", model="tinyllama", type="q8_0", pos=191),
        # the headline: an 8B model generating with 2048 positions of context, f16 and the mix of
        # types most quantized files have
        dict(name="llama3_decode_f16", kind="decode", model="llama3", type="f16", pos=2048),
        dict(name="llama3_decode_q4_k_m", kind="decode", model="llama3", type="q4_k_m", pos=2048),
        # prompts: a short first turn, a ragged 8-bit document, a long one on the 8B model, and a short
        # follow-up turn after 500 positions on the quantized 8B model
        dict(name="tinyllama_prefill_f16", kind="prefill", model="tinyllama", type="f16", n=128, start=0),
        dict(name="tinyllama_prefill_q8_0", kind="prefill", model="tinyllama", type="q8_0", n=777, start=0),
        dict(name="llama3_prefill_f16", kind="prefill", model="llama3", type="f16", n=1024, start=0),
        dict(name="llama3_prefill_q4_k_m", kind="prefill", model="llama3", type="q4_k_m", n=37, start=500),
        # the usual sampler settings over the 8B model's vocabulary
        dict(name="sample_topk_topp", kind="sample", vocab=128256, temperature=0.8, top_k=40, top_p=0.95,
             min_p=0.0, repetition=1.1, context=256),
        # attention as its own call over a long view, and a quantized matrix-vector product on the
        # blocks of a file as they are
        dict(name="attention_32768", kind="attention", seq=32768, nq=32, nkv=8, hd=128),
        dict(name="gemm_q4_k", kind="gemm", type="q4_k", m=1, rows=14336, k=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "decode", "prefill", "prefill", "sample", "attention", "gemm"])
    if kind == "decode":
        model = rng.choice(["tiny", "tinyllama", "tinyllama", "llama3"])
        types = {"tiny": ["f16"], "tinyllama": ["f16", "q8_0", "q4_0", "q4_k", "q5_k", "q6_k", "q4_k_m"],
                 "llama3": ["f16", "q4_k_m", "q6_k"]}[model]
        return dict(kind=kind, model=model, type=rng.choice(types), pos=_log(rng, 1, 500 if model == "tiny" else 2048))
    if kind == "prefill":
        model = rng.choice(["tiny", "tinyllama", "tinyllama", "tinyllama", "llama3"])
        types = {"tiny": ["f16"], "tinyllama": ["f16", "f16", "q8_0", "q4_0", "q4_k", "q5_k", "q6_k", "q4_k_m"],
                 "llama3": ["f16", "q4_k_m"]}[model]
        return dict(kind=kind, model=model, type=rng.choice(types), n=_log(rng, 2, 256 if model == "tiny" else 1024),
                    start=rng.choice([0, 0, _log(rng, 1, 250 if model == "tiny" else 1000)]))
    if kind == "sample":
        top_k, top_p, min_p = rng.choice([(40, 0.95, 0.0), (0, 0.9, 0.0), (0, 1.0, 0.05), (0, 1.0, 0.0), (1, 1.0, 0.0),
                                          (rng.randint(2, 1000), 1.0, 0.0)])
        return dict(kind=kind, vocab=rng.choice([32000, 128256, _log(rng, 500, 128256)]),
                    temperature=round(rng.uniform(0.5, 1.2), 2), top_k=top_k, top_p=top_p, min_p=min_p,
                    repetition=rng.choice([1.0, 1.1]), context=_log(rng, 1, 1024))
    if kind == "attention":
        nq, nkv, hd = rng.choice([(32, 8, 128), (32, 4, 64), (32, 32, 128), (8, 4, 8)])
        return dict(kind=kind, seq=_log(rng, 1, 512 if hd == 8 else 32768 if nkv < 32 else 8192), nq=nq, nkv=nkv, hd=hd)
    rows, k = rng.choice([(6144, 4096), (14336, 4096), (4096, 14336), (5632, 2048), (2048, 5632), (32000, 2048),
                          (_log(rng, 100, 8000), 256 * rng.randint(1, 24))])
    return dict(kind="gemm", type=rng.choice(["f16", "f16", "q8_0", "q4_0", "q4_k", "q5_k", "q6_k"]),
                m=rng.choice([1, 1, _log(rng, 2, 512)]), rows=rows, k=k)


# ------------------------------------------------------------------ weights and inputs (from the seed alone)

def _gen(seed, i):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 100003 + i) % (1 << 60))
    return g


def _q4_k_m(name, layers):
    """The types of a Q4_K_M file: Q6_K output, and Q6_K attn_v / ffn_down in the first and last eighth
    of the layers and every third one between."""
    part = name.split(".")
    if part[0] == "output":
        return "q6_k"
    if len(part) > 2 and part[2] in ("attn_v", "ffn_down"):
        i = int(part[1])
        if i < layers // 8 or i >= 7 * layers // 8 or (i - layers // 8) % 3 == 2:
            return "q6_k"
    return "q4_k"


def _tensors(case):
    """(name, rows, cols, type) of every tensor of the case's model; norms have rows 1."""
    c = MODELS[case["model"]]
    d, f, kvd = c["dim"], c["ffn"], c["dim"] // c["n_heads"] * c["n_kv_heads"]
    out = [("token_embd.weight", c["vocab"], d), ("output_norm.weight", 1, d), ("output.weight", c["vocab"], d)]
    for i in range(c["n_layers"]):
        b = "blk.%d." % i
        out += [(b + "attn_norm.weight", 1, d), (b + "attn_q.weight", d, d), (b + "attn_k.weight", kvd, d),
                (b + "attn_v.weight", kvd, d), (b + "attn_output.weight", d, d), (b + "ffn_norm.weight", 1, d),
                (b + "ffn_gate.weight", f, d), (b + "ffn_up.weight", f, d), (b + "ffn_down.weight", d, f)]
    t = case["type"]
    return [(n, r, k, "norm" if r == 1 else _q4_k_m(n, c["n_layers"]) if t == "q4_k_m" else t) for n, r, k in out]


def _f16_bytes(x):
    return x.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _tensor(rows, cols, kind, g):
    """One tensor on the GPU: f16 values, or the GGUF blocks [rows, blocks, bytes] of a quantized one
    (weights of standard deviation near STD)."""
    if kind == "norm":
        return 1.0 + STD * torch.randn(1, cols, generator=g, device="cuda").half()
    if kind == "f16":
        return torch.randn(rows, cols, generator=g, device="cuda", dtype=torch.float16) * STD
    elems, size = BLOCK[kind]
    nb = cols // elems
    b = torch.randint(0, 256, (rows, nb, size), generator=g, device="cuda", dtype=torch.uint8)
    u = 0.5 + torch.rand(rows, nb, generator=g, device="cuda")
    if kind in ("q4_0", "q8_0"):
        b[..., 0:2] = _f16_bytes(u * (STD / (4.61 if kind == "q4_0" else 73.6)))
        if kind == "q8_0":
            b[..., 2:].masked_fill_(b[..., 2:] == 128, 129)  # quants of -127 .. 127
    elif kind in ("q4_k", "q5_k"):
        sd, mid = (4.61, 7.5) if kind == "q4_k" else (9.23, 15.5)
        d = (u * (STD / (40.0 * sd))).half()
        s = torch.randint(16, 64, (rows, nb, 8), generator=g, device="cuda", dtype=torch.uint8)
        b[..., 0:2] = _f16_bytes(d)
        b[..., 2:4] = _f16_bytes(d.float() * mid)
        # the min of a sub-block equals its scale, so that weights centre on 0
        b[..., 4:8] = s[..., :4] | ((s[..., 4:] >> 4) << 6)
        b[..., 8:12] = b[..., 4:8]
        b[..., 12:16] = (s[..., 4:] & 15) | ((s[..., 4:] & 15) << 4)
    else:
        b[..., 192:208] = torch.randint(16, 48, (rows, nb, 16), generator=g, device="cuda", dtype=torch.uint8)
        b[..., 208:210] = _f16_bytes(u * (STD / (32.0 * 18.5)))
    return b


def _tokens(case, count, seed):
    g = torch.Generator()
    g.manual_seed(int(seed) + 17)
    return torch.randint(0, MODELS[case["model"]]["vocab"], (count,), generator=g).tolist()


_held = {}


def _host(t):
    """The tensor's bytes in one pinned host buffer, kept for the next tensor."""
    n = t.numel() * t.element_size()
    if _held.get("pin") is None or _held["pin"].numel() < n:
        _held["pin"] = torch.empty(max(n, 64 << 20), dtype=torch.uint8, pin_memory=True)
    h = _held["pin"][:n]
    h.copy_(t.contiguous().view(-1).view(torch.uint8))
    return h.numpy()


def _model(case, seed, rows):
    """A context and the case's model in it with `rows` KV rows, every weight uploaded."""
    gc.collect()
    c = MODELS[case["model"]]
    ts = _tensors(case)
    size = sum((r + 15) // 16 * 16 * k * {"norm": 2.0, "f16": 2.0, "q8_0": 1.07}.get(t, 0.9) for _, r, k, t in ts)
    kvd = c["dim"] // c["n_heads"] * c["n_kv_heads"]
    well = size + 4 * c["n_layers"] * rows * kvd + (1 << 30)
    ctx = A.Context(int(well))
    cfg = A.ModelConfig(c["dim"], c["n_layers"], c["n_heads"], c["n_kv_heads"], c["ffn"], c["vocab"], rows, EPS,
                        c["theta"], 1, -1)
    kinds = {t for _, _, _, t in ts} - {"norm"}
    if len(kinds) == 1:
        m = A.Model.create(ctx, cfg, TYPES[kinds.pop()])
    else:
        m = A.Model.create_mixed(ctx, cfg, {n: TYPES[t] for n, _, _, t in ts if t != "norm"})
    blocks = {"q4_0": A.Q4_0Tensor, "q8_0": A.Q8_0Tensor, "q4_k": A.Q4_KTensor, "q5_k": A.Q5_KTensor, "q6_k": A.Q6_KTensor}
    for i, (n, r, k, t) in enumerate(ts):
        w = _tensor(r, k, t, _gen(seed, i))
        h = w.cpu().numpy() if t == "q8_0" else _host(w)  # Q8_0 blocks are taken apart on the host: slow from pinned memory
        m.set_tensor(n, h.view(np.float16).reshape(r, k) if t in ("norm", "f16") else blocks[t](h, r, k))
    return ctx, m


def _ops():
    """The context of the calls that need no model: one for the program, as its host keeps it."""
    if "ctx" not in _held:
        _held["ctx"] = A.Context(1 << 30)
    return _held["ctx"]


def _wrap(t):
    """A tensor of the library over a torch tensor's memory."""
    r, k = (1, t.numel()) if t.dim() == 1 else t.shape
    return A.Tensor(_ops(), t.data_ptr(), r, k)


def _inputs(case, seed):
    if case["kind"] == "sample":
        x = torch.randn(case["vocab"], generator=_gen(seed, 0), device="cuda") * 2.5
        g = torch.Generator()
        g.manual_seed(int(seed) + 17)
        return x.half(), torch.randint(0, case["vocab"], (case["context"],), generator=g).tolist()
    if case["kind"] == "attention":
        def rnd(i, *s):
            return torch.randn(*s, generator=_gen(seed, i), device="cuda", dtype=torch.float16)
        w = case["nkv"] * case["hd"]
        return rnd(0, case["nq"] * case["hd"]), rnd(1, case["seq"], w), rnd(2, case["seq"], w)
    a = torch.randn(case["m"], case["k"], generator=_gen(seed, 0), device="cuda", dtype=torch.float16)
    return a, _tensor(case["rows"], case["k"], case["type"], _gen(seed, 1))


# ------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    if case["kind"] == "decode":
        toks = _tokens(case, case["pos"] + 1, seed)
        ctx, m = _model(case, seed, case["pos"] + 65)
        m.prefill(toks[:-1], 0)
        m.forward_pass(toks, case["pos"])
        return dict(kind="decode", ctx=ctx, m=m, token=toks[-1:], pos=case["pos"])
    if case["kind"] == "prefill":
        toks = _tokens(case, case["start"] + case["n"], seed)
        ctx, m = _model(case, seed, case["start"] + case["n"] + 64)
        if case["start"]:
            m.prefill(toks[:case["start"]], 0)
        return dict(kind="prefill", ctx=ctx, m=m, tokens=toks[case["start"]:], start=case["start"])
    ins = _inputs(case, seed)
    s = dict(kind=case["kind"], held=ins)
    if case["kind"] == "sample":
        s.update(logits=_wrap(ins[0]), context=ins[1], seed=(int(seed) * 7919 + 1) % (1 << 60),
                 cfg=A.SamplerConfig(case["temperature"], case["top_k"], case["top_p"], case["min_p"], case["repetition"]))
    elif case["kind"] == "attention":
        s["out"] = torch.zeros_like(ins[0])
        s["args"] = [_wrap(t) for t in (*ins, s["out"])] + [case["seq"], case["hd"], case["nq"], case["nkv"]]
    else:
        s["out"] = torch.zeros(case["m"], case["rows"], device="cuda", dtype=torch.float16)
        s.update(type=TYPES[case["type"]], a=_wrap(ins[0]), c=_wrap(s["out"]), rows=case["rows"])
        if case["type"] == "f16":
            s["b"] = _wrap(ins[1])
    torch.cuda.synchronize()
    return s


def run(state):
    if state["kind"] == "decode":
        token = state["m"].forward_pass(state["token"], state["pos"])
        logits = state["m"].logits()
        return {"logits": logits, "best": float(logits[token])}  # the greedy token's logit: near ties may change the index
    if state["kind"] == "prefill":
        token = state["m"].prefill(state["tokens"], state["start"])
        logits = state["m"].logits()
        return {"logits": logits, "best": float(logits[token])}
    if state["kind"] == "sample":
        rng = A.RuneRNG(state["seed"])
        token = A.sample_token(_ops(), state["logits"], state["cfg"], rng, state["context"])
        return {"token": token, "rng": rng.state >> 1}
    if state["kind"] == "attention":
        A.flash_attention_gqa(_ops(), *state["args"])
    elif state["type"] == TYPES["f16"]:
        A.gemm_f16(_ops(), state["a"], state["b"], state["c"])
    else:
        A.gemm_quant(_ops(), state["a"], state["held"][1].data_ptr(), state["type"], state["rows"], state["c"])
    return state["out"]


# ------------------------------------------------------------------ what the path cannot do without

def _bytes(rows, cols, kind):
    return 2 * rows * cols if kind in ("norm", "f16") else rows * cols // BLOCK[kind][0] * BLOCK[kind][1]


def work(case):
    if case["kind"] in ("decode", "prefill"):
        c = MODELS[case["model"]]
        n, at = (1, case["pos"]) if case["kind"] == "decode" else (case["n"], case["start"])
        kvd = c["dim"] // c["n_heads"] * c["n_kv_heads"]
        ts = _tensors(case)
        layer = [t for t in ts if t[0] not in ("token_embd.weight", "output.weight")]
        embd = [t for t in ts if t[0] == "token_embd.weight"][0]
        head = [t for t in ts if t[0] == "output.weight"][0]
        by = sum(_bytes(r, k, t) for _, r, k, t in layer) + _bytes(*head[1:]) + _bytes(min(n, embd[1]), *embd[2:])
        by += 4 * c["n_layers"] * kvd * (at + n) + 2 * c["vocab"]
        keys = n * at + n * (n + 1) // 2
        fl = 2 * n * sum(r * k for _, r, k, t in layer if t != "norm") + 2 * head[1] * head[2] + 4 * c["n_layers"] * c["dim"] * keys
        return {"bytes": by, "flops": fl}
    if case["kind"] == "sample":
        return {"bytes": 2 * case["vocab"] + 8 * case["context"], "flops": 0}
    if case["kind"] == "attention":
        kv = case["seq"] * case["nkv"] * case["hd"]
        return {"bytes": 4 * kv + 4 * case["nq"] * case["hd"], "flops": 4 * case["seq"] * case["nq"] * case["hd"]}
    m, n, k = case["m"], case["rows"], case["k"]
    return {"bytes": _bytes(n, k, case["type"]) + 2 * m * (k + n), "flops": 2 * m * n * k}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    if case["kind"] in ("decode", "prefill"):
        # f16 activations and cache through 5 to 32 layers: the logits measured 0.0006-0.0012, 0.004-0.006 and
        # 0.010-0.014 off 64 bits (2-norm); two implementations differ by the sum of two such errors
        return {"tiny": {"rel": 0.004, "max": 0.03}, "tinyllama": {"rel": 0.02, "max": 0.12},
                "llama3": {"rel": 0.03, "max": 0.2}}[case["model"]]
    # one f16 rounding of an f32 sum: measured 0.0002 off 64 bits
    return {"rel": 0.001, "max": 0.01}


# ------------------------------------------------------------------ the same in 64 bits

def _dequant(b, kind):
    """f64 weights of a tensor; a quantized type's weights are f16 by its own rule."""
    if kind in ("norm", "f16"):
        return b.double()
    rows, nb = b.shape[:2]

    def f16(i):
        return b[..., i:i + 2].contiguous().view(torch.float16).double()  # [rows, nb, 1]

    def half(x):
        return x.to(torch.float16).double()

    if kind == "q8_0":
        w = b[..., 2:].contiguous().view(torch.int8).double() * f16(0)
    elif kind == "q4_0":
        w = (torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8.0) * f16(0)
    elif kind in ("q4_k", "q5_k"):
        s = b[..., 4:16]
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
        qs = b[..., 16:] if kind == "q4_k" else b[..., 48:]
        qs = qs.reshape(rows, nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 3).reshape(rows, nb, 8, 32)
        if kind == "q5_k":
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 1, 8, 1)
            q = q | (((b[..., 16:48].unsqueeze(2) >> bit) & 1) << 4)
        w = half(f16(0) * sc).unsqueeze(-1) * q.double() - half(f16(2) * mn).unsqueeze(-1)
    else:
        ql, qh = b[..., 0:128].reshape(rows, nb, 2, 2, 32), b[..., 128:192].reshape(rows, nb, 2, 1, 32)
        lo = torch.stack([ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4, ql[..., 1, :] >> 4], 3)
        sh = (2 * torch.arange(4, device=b.device, dtype=torch.uint8)).view(1, 1, 1, 4, 1)
        q = (lo | (((qh >> sh) & 3) << 4)).double() - 32.0
        a = half(f16(208) * b[..., 192:208].contiguous().view(torch.int8).double())
        w = a.unsqueeze(-1) * q.reshape(rows, nb, 16, 16)
    return half(w).reshape(rows, -1)


def _exact_logits(case, seed, toks):
    c = MODELS[case["model"]]
    ts = {n: (i, r, k, t) for i, (n, r, k, t) in enumerate(_tensors(case))}

    def w(name):
        i, r, k, t = ts[name]
        return _dequant(_tensor(r, k, t, _gen(seed, i)), t)

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w(name)

    hd, nh, nkv, n = c["dim"] // c["n_heads"], c["n_heads"], c["n_kv_heads"], len(toks)
    pos = torch.arange(n, device="cuda", dtype=torch.float64)
    ang = pos[:, None] * c["theta"] ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    x = w("token_embd.weight")[torch.tensor(toks, device="cuda")]
    hide = torch.ones(n, n, device="cuda", dtype=torch.bool).triu(1)
    for i in range(c["n_layers"]):
        b = "blk.%d." % i
        h = norm(x, b + "attn_norm.weight")
        q = rope((h @ w(b + "attn_q.weight").T).view(n, nh, hd))
        k = rope((h @ w(b + "attn_k.weight").T).view(n, nkv, hd))
        v = (h @ w(b + "attn_v.weight").T).view(n, nkv, hd)
        att = torch.empty(n, nh, hd, device="cuda", dtype=torch.float64)
        for j in range(nh):
            g = j // (nh // nkv)
            p = (q[:, j] @ k[:, g].T / math.sqrt(hd)).masked_fill(hide, -math.inf).softmax(-1)
            att[:, j] = p @ v[:, g]
        x = x + att.view(n, -1) @ w(b + "attn_output.weight").T
        h = norm(x, b + "ffn_norm.weight")
        h = torch.nn.functional.silu(h @ w(b + "ffn_gate.weight").T) * (h @ w(b + "ffn_up.weight").T)
        x = x + h @ w(b + "ffn_down.weight").T
    return norm(x[-1:], "output_norm.weight")[0] @ w("output.weight").T


def exact(case, seed):
    if case["kind"] == "sample":
        return None  # whole values
    if case["kind"] in ("decode", "prefill"):
        count = case["pos"] + 1 if case["kind"] == "decode" else case["start"] + case["n"]
        logits = _exact_logits(case, seed, _tokens(case, count, seed)).cpu().numpy()
        return {"logits": logits, "best": None}  # (one rounded value: its error is a matter of chance)
    if case["kind"] == "attention":
        q, k, v = (t.double() for t in _inputs(case, seed))
        nq, nkv, hd = case["nq"], case["nkv"], case["hd"]
        q, k, v = q.view(nkv, nq // nkv, hd), k.view(-1, nkv, hd), v.view(-1, nkv, hd)
        p = (torch.matmul(q, k.permute(1, 2, 0).contiguous()) / math.sqrt(hd)).softmax(-1)
        return torch.matmul(p, v.permute(1, 0, 2).contiguous()).reshape(-1)
    a, b = _inputs(case, seed)
    return a.double() @ _dequant(b, case["type"]).T
