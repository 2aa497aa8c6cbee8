"""The calls that programs built on ``rwkvtune_amd`` spend their GPU time in, at the sizes they make them.

``listed()`` names twelve cases, ``draw(rng)`` gives more of the same ranges; ``prepare`` makes the inputs and
whatever a program keeps between calls (model, state pool, operator), ``run`` is one pass through the public entry
points, ``exact`` the same pass in float64 with plain torch.

Kinds of case (``case["kind"]``):

``model``    a model forward.  ``T = 0``: one decode step over ``rows`` live slots (``forward_pooled``, what a rollout
             repeats per generated token).  ``T = 1``: one interactive token (``forward_with_state``).  ``T > 1``: the
             prompt of a generation (``forward``, logits of the last position).
``wkv``      the inference WKV7 operator on a state pool: ``T = 1`` is the decode step (``wkv7_decode``), ``hi = 0`` a
             uniform batch through the loaded operator, otherwise a ragged prefill of lengths U(T, hi)
             (``wkv7_prefill``).
``train``    forward and backward of the training WKV7 operator; ``state``: the infinite-context operator with an
             initial state, a final state and both their gradients.
``sample``   one batched sampling step over logits rows.
``logp``     the log-probability gather over logits rows (GRPO's recompute after a rollout).
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import rwkvtune_amd as rt
from rwkvtune_amd import operators as wkv
from rwkvtune_amd.model import PRESETS, StatePool

N = 64
V = 65536
DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEV = "cuda"


def listed():
    return [
        # one token of an interactive session on the small model: every launch of 12 layers, almost no work in each
        dict(name="chat_token", kind="model", preset="rwkv7-0.1b", layers=12, rows=1, T=1, dtype="bf16"),
        # two layers and the head of a rollout's decode step, 200 of 256 slots live
        dict(name="rollout_step", kind="model", preset="rwkv7-1.5b", layers=2, rows=200, T=0, dtype="bf16"),
        # two layers of a prompt's prefill before an interactive generation
        dict(name="prompt_block", kind="model", preset="rwkv7-1.5b", layers=2, rows=1, T=1000, dtype="bf16"),
        # the isolated decode step of the benchmark: 256 slots, 32 heads
        dict(name="wkv_step", kind="wkv", seqs=256, T=1, hi=0, heads=32, dtype="bf16"),
        # one prompt's time-mix in one layer
        dict(name="wkv_prompt", kind="wkv", seqs=1, T=1000, hi=1000, heads=32, dtype="bf16"),
        # the benchmark's ragged prefill of a rollout batch
        dict(name="wkv_ragged", kind="wkv", seqs=64, T=64, hi=2048, heads=32, dtype="bf16"),
        # the parity configuration: four 128-token prompts in float32
        dict(name="wkv_fp32", kind="wkv", seqs=4, T=128, hi=0, heads=12, dtype="fp32"),
        # one layer of a small fine-tuning run, one short sample per step
        dict(name="train_short", kind="train", batch=1, T=512, heads=12, state=False, dtype="bf16"),
        # one layer of the 1.5B training step
        dict(name="train_layer", kind="train", batch=8, T=4096, heads=32, state=False, dtype="bf16"),
        # one chunk of a long document under infinite-context training
        dict(name="train_infctx", kind="train", batch=2, T=1000, heads=32, state=True, dtype="bf16"),
        # the sampler of a full rollout step
        dict(name="sample_rows", kind="sample", rows=256, top_p=0.95, top_k=0, dtype="bf16"),
        # log-probabilities of half a chunk of completion tokens
        dict(name="logp_rows", kind="logp", rows=4096, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["model", "wkv", "wkv", "train", "train", "sample", "logp"])
    if kind == "model":
        preset, layers = rng.choice([("rwkv7-0.1b", 12), ("rwkv7-0.4b", 4), ("rwkv7-1.5b", 2)])
        T = rng.choice([0, 1, 2])
        T = T if T < 2 else _log(rng, 16, 1024)
        rows = _log(rng, 1, 256) if T == 0 else rng.randint(1, 4)
        return dict(kind=kind, preset=preset, layers=layers, rows=rows, T=T, dtype="bf16")
    if kind == "wkv":
        heads = rng.choice([12, 16, 32, 40, 64])
        form = rng.choice(["step", "uniform", "ragged", "ragged"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        if form == "step":
            return dict(kind=kind, seqs=_log(rng, 1, 256), T=1, hi=0, heads=heads, dtype=dtype)
        if form == "uniform":
            return dict(kind=kind, seqs=rng.randint(1, 8), T=_log(rng, 16, 2048), hi=0, heads=heads, dtype=dtype)
        lo = _log(rng, 16, 1024)
        return dict(kind=kind, seqs=_log(rng, 1, 64), T=lo, hi=_log(rng, lo, 2048), heads=heads, dtype=dtype)
    if kind == "train":
        state = rng.choice([False, False, True])
        T = _log(rng, 64, 4096)
        if not state:
            T = (T + 15) // 16 * 16  # the standard operator takes multiples of 16
        dtype = rng.choice(["bf16", "bf16", "fp32"]) if state else "bf16"
        return dict(kind=kind, batch=rng.randint(1, 8), T=T, heads=rng.choice([12, 16, 32]), state=state, dtype=dtype)
    if kind == "sample":
        top_p, top_k = rng.choice([(0.95, 0), (0.85, 50), (1.0, 0), (0.7, 0)])
        return dict(kind=kind, rows=_log(rng, 1, 256), top_p=top_p, top_k=top_k, dtype=rng.choice(["bf16", "bf16", "fp32"]))
    return dict(kind=kind, rows=_log(rng, 64, 8192), dtype=rng.choice(["bf16", "bf16", "fp32"]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEV)


def _wkv_inputs(g, shape, heads, dtype):
    """r, w, k, v, a, b of ``(*shape, heads * 64)``: raw decays in the range the model's w0 / LoRA produce, a = -kk and
    b = kk * iclr with kk of unit length per head."""
    r, k, v = (_randn(g, *shape, heads * N) for _ in range(3))
    w = -6.0 + 5.4 * _rand(g, *shape, heads * N)
    kk = F.normalize(_randn(g, *shape, heads, N), dim=-1).reshape(*shape, heads * N)
    b = kk * _rand(g, *shape, heads * N)
    return [x.to(dtype) for x in (r, w, k, v, -kk, b)]


def _lengths(case):
    """The ragged lengths of a case: a fixed draw per case, so that its work does not depend on the seed."""
    if case["hi"] <= case["T"]:
        return [case["T"]] * case["seqs"]
    g = torch.Generator().manual_seed(2)
    return torch.randint(case["T"], case["hi"] + 1, (case["seqs"],), generator=g).tolist()


def _dims(case):
    p = PRESETS[case["preset"]]
    C = p["n_embd"]
    cfg = rt.RWKV7Config(**{**p, "n_layer": case["layers"], "vocab_size": V})
    return cfg, C, C // N


def _weights(case, seed):
    """State dict of a model of the case's architecture: matrices N(0, (0.5 / sqrt(fan_in))^2), per-channel vectors in
    the ranges of a trained layer."""
    cfg, C, H = _dims(case)
    dw, da, dv, dg = cfg.lora_dims()
    g = _gen(seed)
    dt = DTYPE[case["dtype"]]
    sd = {}

    def mat(name, out, inp, fan=None):
        sd[name] = (_randn(g, out, inp) * (0.5 / math.sqrt(fan or inp))).to(dt)

    def vec(name, mid, spread, shape=(C,)):
        sd[name] = (mid + spread * (2 * _rand(g, *shape) - 1)).to(dt)

    def norm(name):
        vec(name + ".weight", 1.0, 0.2)
        vec(name + ".bias", 0.0, 0.2)

    sd["emb.weight"] = _randn(g, V, C).to(dt)
    for i in range(case["layers"]):
        p = f"blocks.{i}."
        for ln in ["ln1", "ln2"] + (["ln0"] if i == 0 else []):
            norm(p + ln)
        for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g"):
            vec(p + "att." + n, 0.5, 0.5, (1, 1, C))
        vec(p + "att.w0", -3.0, 3.0, (1, 1, C))
        vec(p + "att.a0", 0.0, 0.5, (1, 1, C))
        vec(p + "att.k_k", 0.7, 0.1, (1, 1, C))
        vec(p + "att.k_a", 1.0, 0.1, (1, 1, C))
        vec(p + "att.r_k", 0.0, 0.1, (H, N))
        for n, d in (("w", dw), ("a", da), ("g", dg)) + ((("v", dv),) if i > 0 else ()):
            mat(p + f"att.{n}1", C, d, fan=C)
            mat(p + f"att.{n}2", d, C, fan=d)
        if i > 0:
            vec(p + "att.v0", 0.7, 0.2, (1, 1, C))
        for n in ("receptance", "key", "value", "output"):
            mat(p + f"att.{n}.weight", C, C)
        norm(p + "att.ln_x")
        vec(p + "ffn.x_k", 0.5, 0.5, (1, 1, C))
        mat(p + "ffn.key.weight", 4 * C, C)
        mat(p + "ffn.value.weight", C, 4 * C)
    norm("ln_out")
    mat("head.weight", V, C)
    return cfg, sd


def _model_inputs(case, seed):
    """Tokens and recurrent state (float32: kv [L, rows, H, 64, 64], att_x and ffn_x [L, rows, C]) of a model case."""
    _, C, H = _dims(case)
    L, rows, T = case["layers"], case["rows"], case["T"]
    g = _gen(seed + 7919)
    tokens = torch.randint(1, V - 6, (rows, max(T, 1)), generator=g, device=DEV)
    if T > 1:
        return tokens, None
    return tokens, (0.1 * _randn(g, L, rows, H, N, N), _randn(g, L, rows, C), _randn(g, L, rows, C))


def _op_inputs(case, seed):
    """Inputs of a ``wkv`` case: r, w, k, v, a, b and the state pool."""
    g = _gen(seed)
    H, n = case["heads"], case["seqs"]
    if case["T"] == 1:
        shape = (n,)
    elif case["hi"] == 0:
        shape = (n, case["T"])
    else:
        shape = (sum(_lengths(case)),)
    return _wkv_inputs(g, shape, H, DTYPE[case["dtype"]]), 0.1 * _randn(g, n, H, N, N)


def _train_inputs(case, seed):
    g = _gen(seed)
    B, T, H = case["batch"], case["T"], case["heads"]
    dt = DTYPE[case["dtype"]]
    xs = _wkv_inputs(g, (B, T), H, dt)
    dy = _randn(g, B, T, H * N).to(dt)
    s0 = 0.1 * _randn(g, B, H, N, N) if case["state"] else None
    ds = 0.1 * _randn(g, B, H, N, N) if case["state"] else None
    return xs, dy, s0, ds


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "model":
        cfg, sd = _weights(case, seed)
        with torch.device("meta"):
            m = rt.RWKV7Model(cfg)
        m = m.to_empty(device=DEV).to(DTYPE[case["dtype"]])
        m.load_state_dict(sd)
        m.packs()  # the packed weights a program keeps between calls
        tokens, rec = _model_inputs(case, seed)
        st.update(model=m, tokens=tokens)
        rows = case["rows"]
        if case["T"] == 0:
            pool = StatePool(cfg, rows, torch.device(DEV))
            for dst, src in zip((pool.kv, pool.att_x, pool.ffn_x), rec):
                dst.copy_(src)
            st.update(pool=pool, tokens=tokens.reshape(-1), row=torch.arange(rows, dtype=torch.int32, device=DEV))
        elif case["T"] == 1:
            kv, ax, fx = rec
            st["states"] = [{"att_x_prev": ax[i], "att_kv": kv[i], "ffn_x_prev": fx[i]} for i in range(case["layers"])]
    elif kind == "wkv":
        xs, pool = _op_inputs(case, seed)
        st.update(xs=xs, pool=pool)
        if case["T"] > 1 and case["hi"] == 0:
            st["op"] = rt.load_wkv_operator(device="cuda", for_inference=True)
        elif case["T"] > 1:
            cu = [0]
            for n in _lengths(case):
                cu.append(cu[-1] + n)
            st["cu"] = torch.tensor(cu, dtype=torch.int32, device=DEV)
    elif kind == "train":
        xs, dy, s0, ds = _train_inputs(case, seed)
        if case["state"]:
            B, T, H = case["batch"], case["T"], case["heads"]
            xs, dy = [x.view(B, T, H, N) for x in xs], dy.view(B, T, H, N)
            st.update(ds=ds, s0=s0.requires_grad_(True))
        else:
            st["op"] = rt.load_wkv_operator(device="cuda", for_inference=False)
        st.update(xs=[x.requires_grad_(True) for x in xs], dy=dy)
    else:
        # logits as a trained head gives them: a few tokens carry most of the mass
        g = _gen(seed)
        x = 2.0 * _randn(g, case["rows"], V)
        x[:, :64] += 6.0
        st["logits"] = x.to(DTYPE[case["dtype"]])
        if kind == "sample":
            st["seed"] = int(seed)
        else:
            st["index"] = torch.randint(0, V, (case["rows"],), generator=g, device=DEV)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "model":
        m = st["model"]
        if case["T"] == 0:
            pool = st["pool"]
            logits = m.forward_pooled(st["tokens"], st["row"], st["row"], pool, decode=True)
            return {"logits": logits, "kv": pool.kv, "att_x": pool.att_x, "ffn_x": pool.ffn_x}
        if case["T"] == 1:
            logits, states = m.forward_with_state(st["tokens"], st["states"])
            return {"logits": logits, "kv": [s["att_kv"] for s in states]}
        return {"logits": m.forward(st["tokens"], logits_to_keep=1)}
    if kind == "wkv":
        if case["T"] == 1:
            return {"y": wkv.wkv7_decode(st["pool"], None, *st["xs"]), "state": st["pool"]}
        if case["hi"] == 0:
            y, s = st["op"](*st["xs"], state=st["pool"], return_state=True)
            return {"y": y, "state": s}
        return {"y": wkv.wkv7_prefill(st["pool"], None, st["cu"], *st["xs"]), "state": st["pool"]}
    if kind == "train":
        r, w, k, v, a, b = st["xs"]
        if case["state"]:
            y, s = rt.rwkv7_wkv_infctx(w, r, k, v, a, b, state=st["s0"])
            grads = torch.autograd.grad([y, s], [*st["xs"], st["s0"]], [st["dy"], st["ds"]])
            return {"y": y.detach(), "state": s.detach(), "grads": list(grads)}
        y = st["op"](r, w, k, v, a, b)
        return {"y": y.detach(), "grads": list(torch.autograd.grad(y, st["xs"], st["dy"]))}
    if kind == "sample":
        rt.TokenSampler.manual_seed(st["seed"])
        tok, lp = rt.TokenSampler.sample_batch(st["logits"], temperature=1.0, top_p=case["top_p"], top_k=case["top_k"])
        return {"token": tok, "logp": lp}
    return {"logp": rt.selective_log_softmax(st["logits"], st["index"])}


def work(case):
    kind = case["kind"]
    es = 4 if case["dtype"] == "fp32" else 2
    if kind == "model":
        cfg, C, H = _dims(case)
        L, rows, T = case["layers"], case["rows"], case["T"]
        lora = 2 * C * sum(cfg.lora_dims())
        M = rows * max(T, 1)
        params = L * (12 * C * C + lora) + V * C
        state = L * rows * (H * N * N + 2 * C) * 4 * (2 if T < 2 else 1)
        # per token and layer: the projections, and the recurrence's three 64 x 64 products per head
        flops = 2.0 * M * L * (12 * C * C + lora + 3 * H * N * N) + 2.0 * rows * V * C
        return {"bytes": es * (params + M * C + rows * V) + state, "flops": flops}
    if kind == "wkv":
        H, n = case["heads"], case["seqs"]
        tokens = n if case["T"] == 1 else n * case["T"] if case["hi"] == 0 else sum(_lengths(case))
        return {"bytes": 7 * tokens * H * N * es + 2 * n * H * N * N * 4, "flops": 8.0 * tokens * H * N * N}
    if kind == "train":
        tokens, H = case["batch"] * case["T"], case["heads"]
        # six inputs and dy in, y and six gradients out; backward about twice the forward's operations
        states = 4 * case["batch"] * H * N * N * 4 if case["state"] else 0
        return {"bytes": 14 * tokens * H * N * es + states, "flops": 30.0 * tokens * H * N * N}
    if kind == "sample":
        return {"bytes": case["rows"] * (V * es + 12), "flops": 0}
    return {"bytes": case["rows"] * (V * es + 8 + es), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "model":
        return {"rel": 1e-2, "max": 0.2}  # bf16 activations between the kernels of a layer
    if kind in ("wkv", "train"):
        # 16-bit outputs: their rounding; float32: sums of 64 terms carried over the sequence
        rel = {"bf16": 8e-3, "fp16": 1e-3, "fp32": 1e-5}[case["dtype"]]
        return {"rel": rel, "max": 40 * rel}
    if kind == "sample":
        return {"rel": 1e-4, "max": 1e-2, "differ": 0.01}
    return {"rel": 5e-3 if case["dtype"] == "bf16" else 1e-5}


# ---------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------

def _wkv64(r, w, k, v, a, b, S, dy=None, dS=None, seg=64):
    """The recurrence over ``[B, T, H, 64]`` float64 inputs (``w`` the decay's logarithm, <= 0) from ``S [B * H, 64, 64]``:
    ``(y, S_T)``, and with ``dy`` also the gradients of r, log-decay, k, v, a, b and the initial state."""
    B, T, H, _ = r.shape

    def rows(x):
        return x.permute(1, 0, 2, 3).reshape(T, B * H, N).contiguous()

    def back(x):
        return x.view(T, B, H, N).permute(1, 0, 2, 3)

    r, lw, k, v, a, b = (rows(x) for x in (r, w, k, v, a, b))
    wd = lw.exp()
    y, sa = torch.empty_like(r), torch.empty_like(r)

    def step(S, t):
        sa[t] = (S * a[t, :, None, :]).sum(-1)
        return S * wd[t, :, None, :] + v[t, :, :, None] * k[t, :, None, :] + sa[t, :, :, None] * b[t, :, None, :]

    starts = {}
    for t in range(T):
        if dy is not None and t % seg == 0:
            starts[t] = S
        S = step(S, t)
        y[t] = (S * r[t, :, None, :]).sum(-1)
    if dy is None:
        return back(y), S
    dy = rows(dy)
    g = [torch.empty_like(r) for _ in range(6)]
    dS = torch.zeros_like(S) if dS is None else dS
    for t0 in sorted(starts, reverse=True):
        states = [starts[t0]]
        for t in range(t0, min(T, t0 + seg)):
            states.append(step(states[-1], t))
        for t in range(min(T, t0 + seg) - 1, t0 - 1, -1):
            now, before = states[t - t0 + 1], states[t - t0]
            dS = dS + dy[t, :, :, None] * r[t, :, None, :]
            g[0][t] = (now * dy[t, :, :, None]).sum(-2)
            g[1][t] = (dS * before).sum(-2) * wd[t]
            g[2][t] = (dS * v[t, :, :, None]).sum(-2)
            g[3][t] = (dS * k[t, :, None, :]).sum(-1)
            dsa = (dS * b[t, :, None, :]).sum(-1)
            g[4][t] = (before * dsa[:, :, None]).sum(-2)
            g[5][t] = (dS * sa[t, :, :, None]).sum(-2)
            dS = dS * wd[t, :, None, :] + dsa[:, :, None] * a[t, :, None, :]
    return back(y), S, [back(x) for x in g], dS


def _exact_model(case, seed):
    cfg, sd = _weights(case, seed)
    sd = {n: x.double() for n, x in sd.items()}
    _, C, H = _dims(case)
    tokens, rec = _model_inputs(case, seed)
    B, T = tokens.shape
    x = sd["emb.weight"][tokens]
    kvs, axs, fxs, first = [], [], [], None

    def ln(x, name):
        return F.layer_norm(x, (C,), sd[name + ".weight"], sd[name + ".bias"], 1e-5)

    def shifted(h, prev):
        return torch.cat([prev[:, None], h[:, :-1]], 1) - h

    for i in range(case["layers"]):
        p = f"blocks.{i}."
        W = {n[len(p):]: t for n, t in sd.items() if n.startswith(p)}
        kv, ax, fx = (t[i].double() for t in rec) if rec else (
            torch.zeros(B, H, N, N, dtype=torch.float64, device=DEV), *(torch.zeros(B, C, dtype=torch.float64, device=DEV),) * 2)
        if i == 0:
            x = ln(x, p + "ln0")
        h = ln(x, p + "ln1")
        xx = shifted(h, ax)
        axs.append(h[:, -1])
        xr, xw, xk, xv, xa, xg = (h + xx * W["att." + n].view(C) for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g"))
        r, k, v = (q @ W[f"att.{n}.weight"].t() for q, n in ((xr, "receptance"), (xk, "key"), (xv, "value")))
        w = -F.softplus(-(W["att.w0"].view(C) + torch.tanh(xw @ W["att.w1"]) @ W["att.w2"])) - 0.5
        if first is None:
            first = v
        else:
            v = v + (first - v) * torch.sigmoid(W["att.v0"].view(C) + xv @ W["att.v1"] @ W["att.v2"])
        a = torch.sigmoid(W["att.a0"].view(C) + xa @ W["att.a1"] @ W["att.a2"])
        gate = torch.sigmoid(xg @ W["att.g1"]) @ W["att.g2"]
        kk = F.normalize((k * W["att.k_k"].view(C)).view(B, T, H, N), dim=-1)
        k = k * (1 + (a - 1) * W["att.k_a"].view(C))
        r4, k4, v4, a4 = (t.view(B, T, H, N) for t in (r, k, v, a))
        y, S = _wkv64(r4, -torch.exp(w).view(B, T, H, N), k4, v4, -kk, kk * a4, kv.reshape(B * H, N, N))
        kvs.append(S.view(B, H, N, N))
        y = F.group_norm(y.reshape(B * T, C), H, W["att.ln_x.weight"], W["att.ln_x.bias"], eps=64e-5).view(B, T, H, N)
        y = y + (r4 * k4 * W["att.r_k"]).sum(-1, keepdim=True) * v4
        x = x + (y.reshape(B, T, C) * gate) @ W["att.output.weight"].t()
        h = ln(x, p + "ln2")
        xk = h + shifted(h, fx) * W["ffn.x_k"].view(C)
        fxs.append(h[:, -1])
        x = x + torch.relu(xk @ W["ffn.key.weight"].t()) ** 2 @ W["ffn.value.weight"].t()
    logits = ln(x[:, -1:], "ln_out") @ sd["head.weight"].t()
    if case["T"] == 0:
        return {"logits": logits[:, 0], "kv": torch.stack(kvs), "att_x": torch.stack(axs), "ffn_x": torch.stack(fxs)}
    return {"logits": logits, "kv": kvs} if case["T"] == 1 else {"logits": logits}


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _exact_model(case, seed)
    if kind == "wkv":
        xs, pool = _op_inputs(case, seed)
        H, n = case["heads"], case["seqs"]
        xs = [x.double() for x in xs]
        xs[1] = -xs[1].exp()
        S = pool.double().view(n * H, N, N)
        if case["T"] == 1 or case["hi"] == 0:
            y, S = _wkv64(*(x.view(n, -1, H, N) for x in xs), S)
            return {"y": y.reshape(xs[0].shape), "state": S.view(n, H, N, N)}
        # ragged: zero inputs with decay 1 past a sequence's end leave its state alone
        lens = _lengths(case)
        y, S = _wkv64(*(torch.nn.utils.rnn.pad_sequence(x.split(lens), batch_first=True).view(n, -1, H, N) for x in xs), S)
        return {"y": torch.cat([y[i, :m] for i, m in enumerate(lens)]).reshape(-1, H * N), "state": S.view(n, H, N, N)}
    if kind == "train":
        xs, dy, s0, ds = _train_inputs(case, seed)
        B, T, H = case["batch"], case["T"], case["heads"]
        xs = [x.double().view(B, T, H, N) for x in xs]
        lw = xs[1] = -xs[1].exp()
        S = torch.zeros(B * H, N, N, dtype=torch.float64, device=DEV) if s0 is None else s0.double().view(B * H, N, N)
        y, S, g, dS = _wkv64(*xs, S, dy.double().view(B, T, H, N), None if ds is None else ds.double().view(B * H, N, N))
        g[1] = g[1] * lw  # d log-decay / dw = -exp(w)
        if case["state"]:
            return {"y": y, "state": S.view(B, H, N, N), "grads": [*g, dS.view(B, H, N, N)]}
        return {"y": y.reshape(B, T, H * N), "grads": [x.reshape(B, T, H * N) for x in g]}
    if kind == "logp":
        st = prepare(case, seed)
        out = [torch.log_softmax(x.double(), -1).gather(1, i[:, None])[:, 0]
               for x, i in zip(st["logits"].split(512), st["index"].split(512))]
        return {"logp": torch.cat(out)}
    return None  # drawn tokens: no value to be near to
