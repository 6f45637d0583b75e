"""Performance cases of the fp16 batch-1 inference path: decode steps, prompt prefill and the
attention layer on device buffers, through the public entry points of yalm_amd.hip.

A case is one of
  decode   `steps` tokens decoded one after the other behind `start` cached positions: greedy steps
           (the token comes back), the last one a logits step. The tokens fed in are given, so two
           implementations that differ by a rounding still compute the same thing.
  prefill  a prompt of `n` tokens at positions start .. start + n - 1 behind `start` cached ones,
           returning the last token's logits.
  attention  one layer's decode attention over a KV cache in device memory, on the caller's stream.

Model shapes are the 7B benchmark shape (32/8 heads of 128, hidden 14336), the tiny test shape, a
generic 1B-class shape (dim 2048, heads of 64) and a generic 7B shape without grouped heads (32 kv
heads, hidden 11008). Weights are seeded N(0, 0.02) fp16 as in the benchmark, every tensor a slice of
one pool at an offset of its own (odd distances, so that no two tensors' rows line up); caches are
N(0, 1) fp16. A pass returns the logits (and greedy tokens): the K/V entries it writes stay on the
device, as in a user's program, and reach the logits through every later layer and token.
"""
import ctypes
import math

import numpy as np
import torch

from yalm_amd import hip

SHAPES = {
    # name: dim, hidden, layers, heads, kv heads, head_dim, vocab
    "tiny": (256, 768, 4, 8, 2, 32, 32000),
    "1b": (2048, 8192, 16, 32, 8, 64, 32000),
    "7b": (4096, 14336, 32, 32, 8, 128, 32000),
    "7b-mha": (4096, 11008, 32, 32, 32, 128, 32000),
}
THETA, EPS = 1e6, 1e-5
W_STD = 0.02


def _decode(name, shape, start, steps, ctx):
    return {"name": name, "kind": "decode", "shape": shape, "start": start, "steps": steps, "ctx": ctx}


def _prefill(name, shape, n, start, ctx):
    return {"name": name, "kind": "prefill", "shape": shape, "n": n, "start": start, "ctx": ctx}


def listed():
    return [
        # the smallest model the tests run end to end: launches and latency are all there is
        _decode("decode_tiny", "tiny", 41, 8, 512),
        # one layer's attention called from a program that holds its own cache: a mid-length context
        {"name": "attention_5001", "kind": "attention", "heads": 32, "kv_heads": 8, "hd": 128, "kv": 5001, "ctx": 8192},
        # a small model in a chat of some hundred tokens
        _decode("decode_1b", "1b", 700, 4, 4096),
        # the headline: the first tokens after a short prompt
        _decode("decode_short", "7b", 90, 4, 4096),
        # a long conversation or document at the usual 4K context
        _decode("decode_3200", "7b", 3203, 4, 4096),
        # the attention-heavy end: 16K cached tokens
        _decode("decode_16k", "7b", 16390, 2, 16448),
        # a model without grouped heads: four times the cache per token
        _decode("decode_mha", "7b-mha", 900, 2, 4096),
        # a one-line prompt (the benchmark's 32 tokens)
        _prefill("prefill_32", "7b", 32, 0, 4096),
        # an ordinary chat prompt, no multiple of anything
        _prefill("prefill_203", "7b", 203, 0, 4096),
        # the next turn of a long conversation: few new tokens behind many cached ones
        _prefill("prefill_turn", "7b", 61, 3001, 4096),
        # a page of text
        _prefill("prefill_1013", "7b", 1013, 0, 4096),
        # the benchmark's long prompt
        _prefill("prefill_3200", "7b", 3200, 0, 4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "attention"])
    if kind == "attention":
        kv_heads, group = rng.choice([(8, 4), (8, 4), (4, 8), (8, 1), (16, 2), (2, 4)])
        hd = rng.choice([64, 128, 128])
        kv = _log(rng, 20, 30000)
        return {"kind": kind, "heads": kv_heads * group, "kv_heads": kv_heads, "hd": hd, "kv": kv,
                "ctx": -(-(kv + rng.randrange(0, 512)) // 32) * 32}
    shape = rng.choice(["tiny", "1b", "7b", "7b", "7b-mha"])
    if kind == "decode":
        steps = rng.randrange(1, 5)
        most = {"tiny": 500, "1b": 4000, "7b": 16400, "7b-mha": 4000}[shape]
        start = _log(rng, 1, most)
        ctx = 512 if shape == "tiny" else 4096 if start + steps <= 4096 else 16448
        return {"kind": kind, "shape": shape, "start": start, "steps": steps, "ctx": ctx}
    ctx = 512 if shape == "tiny" else 4096
    n = _log(rng, 2, 500 if shape == "tiny" else 3100)
    # half of the prompts open a conversation, half continue one
    start = 0 if rng.random() < 0.5 else _log(rng, 1, ctx - n)
    return {"kind": kind, "shape": shape, "n": n, "start": start, "ctx": ctx}


# ---- inputs ----------------------------------------------------------------------------------
def _cfg(case):
    dim, hidden, layers, heads, kvh, hd, vocab = SHAPES[case["shape"]]
    return dict(dim=dim, hidden_dim=hidden, head_dim=hd, n_layers=layers, n_heads=heads, n_kv_heads=kvh,
                vocab_size=vocab, max_seq_len=case["ctx"], rotary_dim=hd, rope_theta=THETA, norm_eps=EPS,
                qkv_clip=3.4028234663852886e38, act=1)


def _shapes(c):
    qd, kvd = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    yield "model.embed.weight", (c["vocab_size"], c["dim"])
    yield "model.output.weight", (c["vocab_size"], c["dim"])
    for i in range(c["n_layers"]):
        p = f"model.layers.{i}."
        yield p + "attn.wq.weight", (qd, c["dim"])
        yield p + "attn.wk.weight", (kvd, c["dim"])
        yield p + "attn.wv.weight", (kvd, c["dim"])
        yield p + "attn.wo.weight", (c["dim"], qd)
        yield p + "mlp.w1.weight", (c["hidden_dim"], c["dim"])
        yield p + "mlp.w3.weight", (c["hidden_dim"], c["dim"])
        yield p + "mlp.w2.weight", (c["dim"], c["hidden_dim"])


def _pool(n, std, seed, stream):
    """n fp16 draws of N(0, std) on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(2 * int(seed) + stream)
    out = torch.empty(n, dtype=torch.float16, device="cuda")
    for i in range(0, n, 1 << 24):
        m = min(1 << 24, n - i)
        out[i:i + m] = (torch.randn(m, generator=g, device="cuda") * std).half()
    return out


def _cut(pool, k, n):
    """The k-th tensor's slice of the pool: offsets step by an odd prime, modulo the room there is."""
    off = (k * 1299709 + 1) % (pool.numel() - n)
    return pool[off:off + n]


def _weights(c, seed):
    """(pool, {name: (slice number, shape)}, gains): every tensor of the model."""
    names = {name: (k, shape) for k, (name, shape) in enumerate(_shapes(c))}
    most = max(a * b for _, (a, b) in names.values())
    pool = _pool(most + (1 << 22) + 3, W_STD, seed, 0)
    rng = np.random.default_rng(seed)
    gains = {}
    for i in range(c["n_layers"]):
        for n in ("attn.norm.weight", "mlp.norm.weight"):
            gains[f"model.layers.{i}.{n}"] = (1 + 0.1 * rng.standard_normal(c["dim"])).astype(np.float32)
    gains["model.norm.weight"] = (1 + 0.1 * rng.standard_normal(c["dim"])).astype(np.float32)
    return pool, names, gains


def _tokens(c, n, seed):
    return np.random.default_rng([int(seed), 7]).integers(0, c["vocab_size"], n).astype(np.int32)


def _kv_pool(c, seed):
    return _pool(c["n_kv_heads"] * c["head_dim"] * c["max_seq_len"] + (1 << 20) + 3, 1.0, seed, 1)


def _attention_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    n = case["kv_heads"] * case["hd"] * case["ctx"]
    q = torch.randn(case["heads"] * case["hd"], generator=g, device="cuda")
    k = torch.randn(n, generator=g, device="cuda").half()
    v = torch.randn(n, generator=g, device="cuda").half()
    return q, k, v


def prepare(case, seed):
    if case["kind"] == "attention":
        q, k, v = _attention_inputs(case, seed)
        return {"case": case, "q": q, "k": k, "v": v, "out": torch.empty_like(q)}
    c = _cfg(case)
    pool, names, gains = _weights(c, seed)
    host = pool.cpu().numpy().view(np.uint16)
    tensors = dict(gains)
    for name, (k, shape) in names.items():
        tensors[name] = _cut(torch.from_numpy(host.view(np.int16)), k, shape[0] * shape[1]).numpy().view(np.uint16)
    model = hip.HipModel(c, tensors)
    if case["start"] > 0:  # the positions decoded or prefilled earlier
        kv = torch.from_numpy(_kv_pool(c, seed).cpu().numpy().view(np.int16))
        n = c["n_kv_heads"] * c["head_dim"] * c["max_seq_len"]
        for i in range(c["n_layers"]):
            model.set_kv(i, _cut(kv, 2 * i, n).numpy().view(np.uint16), _cut(kv, 2 * i + 1, n).numpy().view(np.uint16))
    n = case["steps"] if case["kind"] == "decode" else case["n"]
    return {"case": case, "model": model, "tokens": _tokens(c, n, seed)}


def run(state):
    case = state["case"]
    if case["kind"] == "attention":
        q, k, v, out = state["q"], state["k"], state["v"], state["out"]
        at = ctypes.c_void_p
        hip._check(hip.lib().yhip_attention_noalloc(
            at(q.data_ptr()), at(k.data_ptr()), at(v.data_ptr()), case["hd"], case["kv"] - 1, case["ctx"],
            case["heads"], case["kv_heads"], 0, THETA, case["hd"], at(out.data_ptr()),
            at(torch.cuda.current_stream().cuda_stream)))
        return out
    model, tokens = state["model"], state["tokens"]
    if case["kind"] == "prefill":
        return model.prefill(tokens, start_pos=case["start"])
    greedy = [model.forward_argmax(int(t), case["start"] + i) for i, t in enumerate(tokens[:-1])]
    logits = model.forward(int(tokens[-1]), case["start"] + len(tokens) - 1)
    return {"greedy": np.array(greedy, np.int64), "logits": logits} if greedy else {"logits": logits}


# ---- what a pass cannot do without --------------------------------------------------------------
def work(case):
    if case["kind"] == "attention":
        kv, hd = case["kv"], case["hd"]
        return {"bytes": 4 * case["kv_heads"] * hd * kv + 8 * case["heads"] * hd, "flops": 4 * case["heads"] * hd * kv}
    c = _cfg(case)
    d, hid, L, V = c["dim"], c["hidden_dim"], c["n_layers"], c["vocab_size"]
    qd, kvd = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    qkv, rest = (qd + 2 * kvd) * d, qd * d + 3 * d * hid  # weights up to the cache, and behind it
    gains = 4 * d * (2 * L + 1)
    if case["kind"] == "decode":  # every step streams the weights and the cache
        total_b = total_f = 0
        for i in range(case["steps"]):
            kv = case["start"] + i + 1
            total_b += 2 * L * (qkv + rest) + gains + 2 * V * d + 2 * d + 4 * L * kvd * (kv + 1)
            total_f += 2 * L * (qkv + rest) + 2 * V * d + 4 * L * qd * kv
        total_b += 4 * V + 4 * (case["steps"] - 1)
        return {"bytes": total_b, "flops": total_f}
    n, start = case["n"], case["start"]
    # only the last row of the last layer is needed beyond its K and V
    rows = n * (L - 1) + 1
    pairs = sum(start + i + 1 for i in range(n)) * (L - 1) + start + n
    flops = 2 * L * n * 2 * kvd * d + 2 * rows * (qd * d + rest) + 4 * qd * pairs + 2 * V * d
    byts = 2 * L * (qkv + rest) + gains + 2 * V * d + 2 * n * d + 4 * V + 4 * n + 4 * L * kvd * (start + n)
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    # about four times the distance measured between the path and exact(): attention 2.3e-7 (fp32 sums,
    # operands split into two halves), decode up to 1.6e-4 (a cache entry that rounds the other way moves
    # an fp16 ulp, which short contexts feel most), prefill up to 6.4e-3 (every activation that enters a
    # matrix product is rounded to fp16, through 32 layers)
    if case["kind"] == "attention":
        return {"rel": 2e-6}
    if case["kind"] == "prefill":
        return {"rel": 2e-2}
    return {"rel": 1e-3, "differ": 0.34}


# ---- 64-bit reference ---------------------------------------------------------------------------
def _norm(x, g):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * g


def _rope(x, pos, hd):
    """x [n][heads * hd]; fp32 angles pos * freq, as the model defines them."""
    j = torch.arange(0, hd, 2, dtype=torch.float32)
    freq = 1.0 / torch.pow(torch.tensor(THETA, dtype=torch.float32), j / hd)
    ang = (pos.float().cpu()[:, None] * freq[None, :]).double().to(x.device)
    cs, sn = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    y = x.view(x.shape[0], -1, hd // 2, 2)
    a, b = y[..., 0], y[..., 1]
    return torch.stack((a * cs - b * sn, a * sn + b * cs), -1).reshape(x.shape)


def _unpack_k(k, kvh, hd, msl):  # [g][hd / 16][t][16] -> [g][t][hd]
    return k.view(kvh, hd // 16, msl, 16).permute(0, 2, 1, 3).reshape(kvh, msl, hd)


def _attend(q, k, v, pos):
    """q [n][G][hd], k [T][hd], v [hd][T]: causal attention of the queries at positions pos."""
    out = torch.empty_like(q)
    t = torch.arange(k.shape[0], device=q.device)
    for h in range(q.shape[1]):
        for i in range(0, q.shape[0], 1024):
            s = (q[i:i + 1024, h] @ k.T) / math.sqrt(q.shape[2])
            s.masked_fill_(t[None, :] > pos[i:i + 1024, None], float("-inf"))
            out[i:i + 1024, h] = torch.softmax(s, -1) @ v.T
    return out


def exact(case, seed):
    if case["kind"] == "attention":
        q, k, v = _attention_inputs(case, seed)
        kvh, hd, ctx, kv = case["kv_heads"], case["hd"], case["ctx"], case["kv"]
        K, V = _unpack_k(k, kvh, hd, ctx)[:, :kv].double(), v.view(kvh, hd, ctx)[:, :, :kv].double()
        q = q.double().view(kvh, -1, hd)
        pos = torch.tensor([kv - 1], device="cuda")
        return torch.cat([_attend(q[g][None], K[g], V[g], pos)[0] for g in range(kvh)]).reshape(-1)
    c = _cfg(case)
    pool, names, gains = _weights(c, seed)
    kvpool = _kv_pool(c, seed) if case["start"] > 0 else None
    hd, kvh, nh, msl, L = c["head_dim"], c["n_kv_heads"], c["n_heads"], c["max_seq_len"], c["n_layers"]
    start, G, kv_n = case["start"], nh // kvh, kvh * hd * msl

    def w(name):
        k, (a, b) = names[name]
        return _cut(pool, k, a * b).view(a, b).double()

    def g(name):
        return torch.from_numpy(gains[name]).cuda().double()

    toks = _tokens(c, case["steps"] if case["kind"] == "decode" else case["n"], seed)
    n = len(toks)  # teacher-forced decode steps are the rows of one causal pass
    pos = torch.arange(start, start + n, device="cuda")
    k, (a, b) = names["model.embed.weight"]
    x = _cut(pool, k, a * b).view(a, b)[torch.from_numpy(toks.astype(np.int64)).cuda()].double()
    for i in range(L):
        p = f"model.layers.{i}."
        xn = _norm(x, g(p + "attn.norm.weight"))
        q = _rope(xn @ w(p + "attn.wq.weight").T, pos, hd).view(n, kvh, G, hd)
        kn = _rope(xn @ w(p + "attn.wk.weight").T, pos, hd).half().double().view(n, kvh, hd)
        vn = (xn @ w(p + "attn.wv.weight").T).half().double().view(n, kvh, hd)
        att = torch.empty_like(q)
        if start:
            K0 = _unpack_k(_cut(kvpool, 2 * i, kv_n), kvh, hd, msl)[:, :start]
            V0 = _cut(kvpool, 2 * i + 1, kv_n).view(kvh, hd, msl)[:, :, :start]
        for gi in range(kvh):
            K, V = kn[:, gi], vn[:, gi].T
            if start:
                K, V = torch.cat((K0[gi].double(), K)), torch.cat((V0[gi].double(), V), 1)
            att[:, gi] = _attend(q[:, gi], K, V, pos)
        x = x + att.reshape(n, nh * hd) @ w(p + "attn.wo.weight").T
        xn = _norm(x, g(p + "mlp.norm.weight"))
        gate = xn @ w(p + "mlp.w1.weight").T
        x = x + (torch.nn.functional.silu(gate) * (xn @ w(p + "mlp.w3.weight").T)) @ w(p + "mlp.w2.weight").T
    if case["kind"] == "prefill":
        x = x[-1:]
    logits = _norm(x, g("model.norm.weight")) @ w("model.output.weight").T
    if case["kind"] == "prefill":
        return logits[-1].cpu()
    out = {"logits": logits[-1].cpu()}
    if n > 1:
        out["greedy"] = logits[:-1].argmax(-1).cpu()
    return out
