"""The work that a user of this framework has it do, as cases that can be
timed and checked: text generation, prompt prefill, whole-context logits, the
training forward's loss, the optimizer step and the row operators, each
through the public entry points (``Engine``, ``GPT``, ``optim``, ``kernels``).

    listed()        the named cases
    draw(rng)       one more case of the same ranges
    prepare(c, s)   what a program holds before the call, made from seed s
    run(state)      one pass; returns its outputs
    work(c)         bytes and operations that a pass cannot do without
    tolerance(c)    how far another correct implementation may be off
    exact(c, s)     the same outputs in 64 bits by plain torch

Models: the 155M shape (d 768, 11 layers, 6 heads of 128), the command line's
default (d 512, 8 layers, 8 heads of 64), the 77M shape (d 512, 4 heads of
128) and the wide shape (d 1536, 12 heads of 128) at three layers, with window
384 on the short layers and the padded GPT-2 vocabulary.
"""

import math

import torch

from attention_nn_amd import kernels, optim
from attention_nn_amd.config import GPTConfig
from attention_nn_amd.engine import Engine
from attention_nn_amd.model import GPT

DEV = "cuda"
VOCAB = 50304
V_TEXT = 50257          # ids that text uses; the rest pads the table
WINDOW = 384
EPS = 1e-6

# name -> (model_dim, heads, layers, full-causal layers)
MODELS = {
    "155m": (768, 6, 11, (4, 10)),
    "cli": (512, 8, 8, (3, 7)),
    "77m": (512, 4, 8, (3, 7)),
    "wide": (1536, 12, 3, (1,)),
}


# ---- the cases ----------------------------------------------------------------

def listed():
    return [
        # one normalisation of a few rows: what a call costs by itself
        {"name": "rms_few_rows", "kind": "rms", "dtype": "f32", "rows": 17, "dim": 512},
        # query rotation of a training batch, with its odd sequence length
        {"name": "rope_batch", "kind": "rope", "dtype": "bf16", "batch": 16, "length": 1023,
         "heads": 6, "head_dim": 128},
        # interactive generation at batch 1: short prompt, greedy
        {"name": "generate_1", "kind": "generate", "model": "155m", "batch": 1, "prompt": 32,
         "steps": 64, "temperature": 0.0, "top_k": 0},
        # the command line's own default model and sampling
        {"name": "generate_cli", "kind": "generate", "model": "cli", "batch": 1, "prompt": 9,
         "steps": 48, "temperature": 0.8, "top_k": 50},
        # a small serving batch, ragged sizes
        {"name": "generate_7", "kind": "generate", "model": "155m", "batch": 7, "prompt": 150,
         "steps": 48, "temperature": 0.8, "top_k": 50},
        # a full serving batch
        {"name": "generate_64", "kind": "generate", "model": "155m", "batch": 64, "prompt": 512,
         "steps": 24, "temperature": 0.8, "top_k": 50},
        # long contexts
        {"name": "generate_long", "kind": "generate", "model": "155m", "batch": 16,
         "prompt": 7680, "steps": 32, "temperature": 0.0, "top_k": 0},
        # the wide model at its batch
        {"name": "generate_wide", "kind": "generate", "model": "wide", "batch": 128,
         "prompt": 1024, "steps": 24, "temperature": 0.8, "top_k": 50},
        # time to the first token of one ordinary prompt
        {"name": "prompt_777", "kind": "generate", "model": "155m", "batch": 1, "prompt": 777,
         "steps": 0, "temperature": 0.8, "top_k": 50},
        # logits of every position of one text (scoring; the recompute-style loop)
        {"name": "score_300", "kind": "logits", "model": "155m", "batch": 1, "length": 300},
        # the training forward at its batch
        {"name": "loss_64x512", "kind": "loss", "model": "155m", "batch": 64, "length": 512},
        # the optimizer step over every parameter
        {"name": "optimizer_155m", "kind": "optim", "model": "155m"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("rms", "relu2", "rope", "generate", "generate", "prompt", "logits",
                       "loss", "optim"))
    if kind in ("rms", "relu2"):
        return {"kind": kind, "dtype": rng.choice(("f32", "bf16")),
                "rows": _log_int(rng, 1, 65536), "dim": rng.choice((512, 768, 1536, 3072, 100, 129))}
    if kind == "rope":
        heads, hd = rng.choice(((8, 64), (4, 128), (6, 128), (12, 128), (3, 36)))
        return {"kind": kind, "dtype": rng.choice(("f32", "bf16")), "batch": _log_int(rng, 1, 32),
                "length": _log_int(rng, 1, 1024), "heads": heads, "head_dim": hd}
    if kind == "optim":
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "wd": rng.choice((0.6, 1.2, 2.4)),
                "momentum": round(rng.uniform(0.85, 0.95), 4)}
    model = rng.choice(sorted(MODELS))
    if kind in ("logits", "loss"):
        length = _log_int(rng, 1 if kind == "logits" else 16, 1024)
        rows = 2048 if kind == "logits" else 16384
        return {"kind": kind, "model": model, "batch": _log_int(rng, 1, max(1, rows // length)),
                "length": length}
    temp = rng.choice((0.0, 0.7, 0.8, 1.0))
    prompt = _log_int(rng, 2, 1000)
    batch = _log_int(rng, 1, min(128, max(1, 32768 // prompt)))
    return {"kind": "generate", "model": model, "batch": batch, "prompt": prompt,
            "steps": 0 if kind == "prompt" else _log_int(rng, 4, 24), "temperature": temp,
            "top_k": 0 if temp == 0.0 else rng.choice((0, 1, 40, 50, 200))}


# ---- inputs -------------------------------------------------------------------

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + stream) % (1 << 62))
    return g


def _config(name, seq_len=1024):
    d, H, L, longs = MODELS[name]
    return GPTConfig(vocab_size=VOCAB, num_layers=L, num_heads=H, model_dim=d, seq_len=seq_len,
                     window=WINDOW, long_layers=longs)


def _params(name, seed):
    """fp32 parameters on the device: the initialisation's distributions for
    the matrices, head and lambdas away from their initial values."""
    d, H, L, _ = MODELS[name]
    g = _gen(seed, 1)
    bound = math.sqrt(3) * 0.5 * d ** -0.5

    def uni(lo, hi, *shape):
        return torch.empty(shape, device=DEV).uniform_(lo, hi, generator=g)

    def normal(std, *shape):
        return torch.empty(shape, device=DEV).normal_(0.0, std, generator=g)

    return {
        "embed": normal(0.02, VOCAB, d),
        "lm_head": normal(0.03, d, VOCAB),
        "attn_bank": uni(-bound, bound, L, 4, d, d),
        "fc_bank": uni(-bound, bound, L, d, 4 * d),
        "proj_bank": uni(-bound, bound, L, 4 * d, d),
        "resid_lambdas": uni(0.95, 1.1, L, 2),
        "post_lambdas": uni(0.7, 1.2, L, 2),
        "x0_lambdas": uni(-0.2, 0.2, L),
        "sa_lambdas": uni(0.4, 1.1, L, 2),
    }


def _ids(seed, stream, *shape):
    return torch.randint(0, V_TEXT, shape, device=DEV, dtype=torch.int32,
                         generator=_gen(seed, stream))


def _rows(case, seed, *shape):
    dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    return torch.empty(shape, device=DEV).normal_(0.0, 1.0, generator=_gen(seed, 2)).to(dt)


def _rope_tables(length, head_dim):
    d4 = head_dim // 4
    freq = (1.0 / 1024.0) ** torch.linspace(0.0, 1.0, d4, device=DEV)
    theta = torch.arange(length, device=DEV, dtype=torch.float32)[:, None] * freq[None, :]
    return torch.cos(theta).contiguous(), torch.sin(theta).contiguous()


def _grads(name, seed):
    g = _gen(seed, 3)
    return {k: torch.empty(v.shape, device=DEV).normal_(0.0, 1e-3, generator=g)
            for k, v in _params(name, seed).items()}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("rms", "relu2"):
        return {"case": case, "x": _rows(case, seed, case["rows"], case["dim"])}
    if kind == "rope":
        cs, sn = _rope_tables(case["length"], case["head_dim"])
        return {"case": case, "cs": cs, "sn": sn,
                "x": _rows(case, seed, case["batch"], case["length"], case["heads"],
                           case["head_dim"])}
    if kind == "optim":
        params = _params(case["model"], seed)
        opt = optim.MuonAdam(params, optim.optimizer_table(), muon_wd=case.get("wd", 1.2))
        return {"case": case, "params": params, "grads": _grads(case["model"], seed), "opt": opt}
    host = {k: v.cpu().numpy() for k, v in _params(case["model"], seed).items()}
    B = case["batch"]
    if kind == "logits":
        gpt = GPT(_config(case["model"]))
        gpt.engine(host, batch=B)                   # weights laid out once, as the class keeps them
        return {"case": case, "gpt": gpt, "params": host,
                "tokens": _ids(seed, 4, B, case["length"]).cpu().numpy()}
    if kind == "loss":
        T = case["length"]
        eng = Engine(_config(case["model"]), host, max_batch=B, max_ctx=T, max_tokens=B * T)
        return {"case": case, "engine": eng, "tokens": _ids(seed, 4, B, T),
                "targets": _ids(seed, 5, B, T)}
    P, S = case["prompt"], case["steps"]
    ctx = max(1024, P + S)
    eng = Engine(_config(case["model"], ctx), host, max_batch=B, max_ctx=ctx, max_tokens=B * P)
    return {"case": case, "engine": eng, "prompt": _ids(seed, 4, B, P),
            "text": _ids(seed, 5, max(S, 1), B),
            "cur": torch.empty(B, device=DEV, dtype=torch.int32)}


# ---- one pass -----------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "rms":
        return kernels.rms(state["x"])
    if kind == "relu2":
        return kernels.relu2(state["x"])
    if kind == "rope":
        return kernels.rope_ht(state["x"], state["cs"], state["sn"])
    if kind == "optim":
        opt = state["opt"]
        # the next step goes on from these parameters, as a training loop does
        state["params"] = opt(state["params"], state["grads"], 1.0, case.get("momentum", 0.95))
        return {"params": state["params"],
                "state": {n: dict(opt.state[n]) for n in state["params"]}}
    if kind == "logits":
        return state["gpt"].logits(state["params"], state["tokens"])
    if kind == "loss":
        mean, rows = state["engine"].forward_loss(state["tokens"], state["targets"], rows=True)
        return {"mean": mean, "rows": rows}
    # generation along a given text, so that the context is the same whatever
    # is drawn: every step samples a token, and the text's goes in next
    eng, cur, S = state["engine"], state["cur"], case["steps"]
    temp, k = case["temperature"], case["top_k"]
    _, first = eng.prefill(state["prompt"], temp, k, 7, 0, want_logits=True)
    if not S:
        return {"prompt": first}
    last = None
    for i in range(S):
        cur.copy_(state["text"][i])
        _, last = eng.decode(cur, temp, k, 7, i + 1, want_logits=i + 1 == S, out=cur)
    return {"prompt": first, "last": last}


# ---- what a pass cannot do without ----------------------------------------------

def _matrices(name):
    d, H, L, _ = MODELS[name]
    return 12 * d * d * L


def _body_flops(name, B, T, start=0):
    """All layers over T tokens per sequence at positions start ..."""
    d, H, L, longs = MODELS[name]
    keys = 0
    for l in range(L):
        for i in range(start, start + T):
            keys += i + 1 if l in longs else min(i + 1, WINDOW)
    return B * (2.0 * _matrices(name) * T + 4.0 * d * keys)


def _step_bytes(name, B, pos):
    """One decode step: weights once, keys and values read and appended."""
    d, H, L, longs = MODELS[name]
    kv = sum(4 * d * (pos + 1 if l in longs else min(pos + 1, WINDOW)) for l in range(L))
    return 2.0 * (_matrices(name) + d * VOCAB) + B * (kv + L * 4 * d + 2 * d + 8)


def work(case):
    kind = case["kind"]
    if kind in ("rms", "relu2"):
        n = case["rows"] * case["dim"]
        return {"bytes": 2.0 * n * (4 if case["dtype"] == "f32" else 2), "flops": 3.0 * n}
    if kind == "rope":
        n = case["batch"] * case["length"] * case["heads"] * case["head_dim"]
        return {"bytes": 2.0 * n * (4 if case["dtype"] == "f32" else 2)
                + 2.0 * case["length"] * case["head_dim"], "flops": 1.5 * n}
    d, H, L, _ = MODELS[case["model"]]
    if kind == "optim":
        muon, adam = _matrices(case["model"]), 2 * VOCAB * d
        flops = 0.0
        for batch, m, n in ((4 * L, d, d), (L, d, 4 * d), (L, 4 * d, d)):
            s, w = min(m, n), max(m, n)
            flops += 5.0 * batch * (4.0 * s * s * w + 2.0 * s ** 3)
        # p, g and the moments read, p and the moments written, in 4 bytes
        return {"bytes": 4.0 * (5 * muon + 7 * adam), "flops": flops}
    B = case["batch"]
    weights = 2.0 * (_matrices(case["model"]) + d * VOCAB)
    if kind in ("logits", "loss"):
        T = case["length"]
        M = B * T
        out = 4.0 * M * VOCAB if kind == "logits" else 8.0 * M
        return {"bytes": weights + M * (4 + 2 * d + 4 * d * L) + out,
                "flops": _body_flops(case["model"], B, T) + 2.0 * d * VOCAB * M}
    P, S = case["prompt"], case["steps"]
    flops = _body_flops(case["model"], B, P + S) + 2.0 * d * VOCAB * B * (S + 1)
    byts = weights + B * P * (4 + 2 * d + 4 * d * L) + 4.0 * B * VOCAB * (2 if S else 1)
    byts += sum(_step_bytes(case["model"], B, P + i) for i in range(S))
    return {"bytes": byts, "flops": flops}


# ---- tolerances -----------------------------------------------------------------

def tolerance(case):
    """About four times the distance from the same in 64 bits, measured: the
    model's logits are 3.4e-4 to 5.4e-4 off (bf16 weights and activations, a
    bf16 logit before the softcap), the loss's rows 7.2e-4, bf16 rows 1.2e-3,
    32-bit rows 5e-8, the updated matrices 2.1e-3 (bf16 orthogonalisation)."""
    kind = case["kind"]
    if kind == "relu2":
        return "exact"
    if kind in ("rms", "rope"):
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "f32" else {"rel": 4.8e-3, "max": 1.6e-2}
    if kind == "optim":
        return {"rel": 8e-3, "max": 0.2}
    if kind == "loss":
        return {"rel": 3e-3, "max": 0.03}
    return {"rel": 2.2e-3, "max": 0.02}


# ---- the same in 64 bits ----------------------------------------------------------

def _rms64(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


def _rope64(x, cs, sn):
    """x (..., T, H, D); pairs (2j, 2j + 1) below D/4 pairs rotated."""
    d4 = x.shape[-1] // 4
    y = x.clone()
    c, s = cs[:, None, :], sn[:, None, :]
    a, b = x[..., 0:2 * d4:2], x[..., 1:2 * d4:2]
    y[..., 0:2 * d4:2] = c * a + s * b
    y[..., 1:2 * d4:2] = c * b - s * a
    return y


class _Model64:
    """The model's forward in 64 bits from its bf16 weights."""

    def __init__(self, name, seed, length):
        self.d, self.H, self.L, self.longs = MODELS[name]
        p = _params(name, seed)

        def b(t):
            return t.to(torch.bfloat16)

        sa = b(p["sa_lambdas"])
        self.embed, self.head = b(p["embed"]), b(p["lm_head"]).double()
        wl = b(p["attn_bank"])
        self.qkv = [(torch.cat([wl[l, 0], wl[l, 1], wl[l, 2]], -1) * sa[l, 0]).double()
                    for l in range(self.L)]
        self.o = [(wl[l, 3] * sa[l, 1]).double() for l in range(self.L)]
        self.fc = [b(p["fc_bank"][l]).double() for l in range(self.L)]
        self.proj = [b(p["proj_bank"][l]).double() for l in range(self.L)]
        self.r, self.p = b(p["resid_lambdas"]).double(), b(p["post_lambdas"]).double()
        self.x0 = b(p["x0_lambdas"]).double()
        cs, sn = _rope_tables(length, self.d // self.H)
        self.cs, self.sn = cs.double(), sn.double()

    def attend(self, q, k, v, long):
        """(H, T, D) each; blocks of queries against the keys they keep."""
        T = q.shape[1]
        out = torch.empty_like(q)
        for a in range(0, T, 1024):
            z = min(a + 1024, T)
            lo = 0 if long else max(0, a - WINDOW + 1)
            kk = k[:, lo:z].transpose(1, 2).contiguous()
            s = torch.matmul(q[:, a:z].contiguous(), kk) * 0.1
            i = torch.arange(a, z, device=DEV)[:, None]
            j = torch.arange(lo, z, device=DEV)[None, :]
            drop = j > i if long else (j > i) | (i - j >= WINDOW)
            s.masked_fill_(drop, float("-inf"))
            out[:, a:z] = torch.matmul(torch.softmax(s, -1), v[:, lo:z].contiguous())
        return out

    def hidden(self, tokens):
        """rms(x) of every position of (T,) ids."""
        T, H, D = tokens.shape[0], self.H, self.d // self.H
        cs, sn = self.cs[:T], self.sn[:T]
        x = x0 = _rms64(self.embed[tokens.long()].double())
        for l in range(self.L):
            qkv = (_rms64(x) @ self.qkv[l]).reshape(T, 3, H, D)
            q, k = (_rope64(_rms64(qkv[:, n]), cs, sn).transpose(0, 1).contiguous() for n in (0, 1))
            v = qkv[:, 2].transpose(0, 1).contiguous()
            y = self.attend(q, k, v, l in self.longs).transpose(0, 1).reshape(T, self.d) @ self.o[l]
            x = self.r[l, 0] * x + self.p[l, 0] * y + self.x0[l] * x0
            h = torch.clamp_min(_rms64(x) @ self.fc[l], 0.0)
            x = self.r[l, 1] * x + self.p[l, 1] * ((h * h) @ self.proj[l])
        return _rms64(x)

    def logits(self, h):
        return 23.0 * torch.sigmoid((h @ self.head + 5.0) / 7.5)


COEF = ((8.156554524902461, -22.48329292557795, 15.878769915207462),
        (4.042929935166739, -2.808917465908714, 0.5000178451051316),
        (3.8916678022926607, -2.772484153217685, 0.5060648178503393),
        (3.285753657755655, -2.3681294933425376, 0.46449024233003106),
        (2.3465413258596377, -1.7097828382687081, 0.42323551169305323))


def _polar64(g):
    x = g.double()
    x = x / (x.norm(dim=(-2, -1), keepdim=True) * 1.02 + 1e-6)
    tall = x.shape[-2] > x.shape[-1]
    if tall:
        x = x.transpose(-2, -1).contiguous()
    for a, b, c in COEF:
        A = torch.matmul(x, x.transpose(-2, -1).contiguous())
        x = a * x + torch.matmul(b * A + c * torch.matmul(A, A), x)
    return x.transpose(-2, -1).contiguous() if tall else x


def _exact_optim(case, seed):
    p, g = _params(case["model"], seed), _grads(case["model"], seed)
    wd, mu = case.get("wd", 1.2), case.get("momentum", 0.95)
    new, state = {}, {}
    for n, rule in optim.optimizer_table().items():
        pv, gv = p[n].double(), g[n].double()
        if rule["optim"] == "adam":
            b1, b2 = rule["adam_betas"]
            lr = 0.008 * rule.get("lr_mul", 1.0)
            m, v = (1 - b1) * gv, (1 - b2) * gv * gv
            u = m / (v.sqrt() + 1e-10) * (lr * math.sqrt(1 - b2) / (1 - b1))
            u = u + torch.where(u * pv > 0, pv * (lr * lr * 0.005 * rule.get("wd_mul", 1.0)), 0.0)
            new[n], state[n] = pv - u, {"m": m, "v": v}
            continue
        rows, cols = pv.shape[-2:]
        lr = 0.023 * math.sqrt(max(1.0, rows / cols))
        buf = (1 - mu) * gv
        u = _polar64(gv + mu * (buf - gv))
        red = -1 if rows >= cols else -2
        mean = (u * u).mean(red, keepdim=True)
        step = torch.rsqrt(torch.clamp_min(0.1 * mean, 1e-10))
        was = u.norm(dim=(-2, -1), keepdim=True)
        u = u * step
        u = u * (was / u.norm(dim=(-2, -1), keepdim=True))
        keep = torch.where(u * pv >= 0, pv * (0.023 * wd * lr), 0.0)
        # the second moment follows the iteration's own bf16 arithmetic, whose
        # singular values differ from the exact iteration's by several percent
        new[n], state[n] = pv - keep - u * lr, {"momentum": buf, "second_mom": None}
    return {"params": new, "state": state}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("rms", "relu2"):
        x = _rows(case, seed, case["rows"], case["dim"]).double()
        return _rms64(x) if kind == "rms" else torch.clamp_min(x, 0.0) ** 2
    if kind == "rope":
        cs, sn = _rope_tables(case["length"], case["head_dim"])
        x = _rows(case, seed, case["batch"], case["length"], case["heads"], case["head_dim"])
        return _rope64(x.double(), cs.double(), sn.double())
    if kind == "optim":
        return _exact_optim(case, seed)
    B = case["batch"]
    if kind in ("logits", "loss"):
        T = case["length"]
        net = _Model64(case["model"], seed, T)
        tokens = _ids(seed, 4, B, T)
        if kind == "logits":
            return torch.stack([net.logits(net.hidden(tokens[b])) for b in range(B)])
        rows = []
        for b, t in enumerate(_ids(seed, 5, B, T)):
            z = net.logits(net.hidden(tokens[b]))
            rows.append(torch.logsumexp(z, -1) - z.gather(-1, t.long()[:, None])[:, 0])
        rows = torch.cat(rows)
        return {"mean": rows.mean(), "rows": rows}
    P, S = case["prompt"], case["steps"]
    net = _Model64(case["model"], seed, P + S)
    prompt, text = _ids(seed, 4, B, P), _ids(seed, 5, max(S, 1), B)
    first, last = [], []
    for b in range(B):
        h = net.hidden(torch.cat([prompt[b], text[:S, b]]))
        first.append(net.logits(h[P - 1]))
        last.append(net.logits(h[-1]))
    out = {"prompt": torch.stack(first)}
    if S:
        out["last"] = torch.stack(last)
    return out
