"""The work that users of this framework have it do, as cases that can be timed and checked.

Three ways in, as the README lists them: the Qwen2.5 harness (decode steps and prompts, int4 and bf16 weights),
models of the registry (Lusadra and Girirax: a prompt and the tokens after it), and the C ABI under the reference's
array class (attention over a cache, f32 products) and under a model file's loader (f16 rows to int4 or bf16).
Sizes are those of bench.py and the tests; `draw` spreads them over the ranges in between. Weights are the seeded
ones that every model class offers, so a case needs no file.
"""
import importlib
import math

import numpy as np
import torch

pkg = importlib.import_module("cpp-tensorlib_amd")
qwen = importlib.import_module("cpp-tensorlib_amd.qwen")
model = importlib.import_module("cpp-tensorlib_amd.model")

QWEN = {"0.5B": qwen.QWEN_05B, "7B": qwen.QWEN_7B}
CONTEXT = {"0.5B": 2304, "7B": 4352}           # what a model is created for
# The folder designs at the sizes of bench.py. Lusadra: heads, key heads, head size and window of the attention; heads,
# key and value size of the linear attention. Girirax (state-space and latent-attention layers in turn): heads, value
# size, state and groups; heads, key, rotated, value size, latent and query rank.
SIZES = {
    "Lusadra": {
        "small": dict(layers=12, vocab=32000, width=896, left=(14, 2, 64, 512), right=(7, 64, 128), ff=4864),
        "medium": dict(layers=8, vocab=32000, width=2048, left=(16, 4, 128, 1024), right=(16, 64, 128), ff=8192),
        "large": dict(layers=4, vocab=32000, width=3584, left=(28, 4, 128, 1024), right=(28, 64, 128), ff=18944)},
    "Girirax": {
        "small": dict(layers=12, vocab=32000, width=896, ssm=(28, 64, 128, 1), latent=(14, 64, 32, 64, 256, 384), ff=4864),
        "medium": dict(layers=8, vocab=32000, width=2048, ssm=(64, 64, 128, 8), latent=(16, 128, 64, 128, 512, 768), ff=8192),
        "large": dict(layers=4, vocab=32000, width=3584, ssm=(112, 64, 128, 8), latent=(28, 128, 64, 128, 512, 1536), ff=18944)},
}
RANK = 16                                        # of Lusadra's decay inputs


def listed():
    return [
        # One token of a small model early in a chat: every launch counts.
        dict(name="qwen0.5b-int4-step", kind="step", model="0.5B", layers=24, fmt="q4", pos=200),
        # A question of a few dozen words to the same model, the ordinary prompt of a chat.
        dict(name="qwen0.5b-bf16-prompt77", kind="prompt", model="0.5B", layers=24, fmt="bf16", tokens=77, pos=0),
        # One token of the 7B model deep in a context: the headline decode.
        dict(name="qwen7b-int4-step-4k", kind="step", model="7B", layers=28, fmt="q4", pos=4095),
        # A full prompt chunk at 7B dimensions, bf16 weights: the matrix cores' case (four of its layers, so that the
        # two forms of the weights of several models fit the card).
        dict(name="qwen7b-bf16-prompt512", kind="prompt", model="7B", layers=4, fmt="bf16", tokens=512, pos=0),
        # A follow-up message of an odd length deeper in a conversation, int4 weights.
        dict(name="qwen7b-int4-prompt301", kind="prompt", model="7B", layers=8, fmt="q4", tokens=301, pos=1500),
        # A chat turn with each of the other two designs: a short prompt and the tokens that follow it.
        dict(name="girirax-small-turn", kind="turn", design="Girirax", size="small", prompt=37, tokens=16),
        dict(name="lusadra-medium-turn", kind="turn", design="Lusadra", size="medium", prompt=150, tokens=16),
        # A document read in: several chunks, the last one ragged or not.
        dict(name="girirax-large-document", kind="turn", design="Girirax", size="large", prompt=2048, tokens=0),
        dict(name="lusadra-large-document", kind="turn", design="Lusadra", size="large", prompt=1001, tokens=0),
        # array::attn_decode at the reference benchmark's 28 heads of their own keys.
        dict(name="attention-28x2048", kind="attention", heads=28, kv_heads=28, dim=128, ctx=2048, kv="f32"),
        # array::dot of two f32 matrices: a ragged batch of rows through a projection.
        dict(name="product-f32-333", kind="product", m=333, n=4864, k=896, ta=False, tb=False),
        # A model file's f16 rows on their way to int4 groups: the 7B gate projection.
        dict(name="load-int4-18944", kind="load", rows=18944, cols=3584, to="q4"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "prompt", "prompt", "turn", "turn", "turn", "attention", "product", "load"])
    if kind in ("step", "prompt"):
        m, fmt = rng.choice(["0.5B", "7B"]), rng.choice(["q4", "bf16"])
        layers = 24 if m == "0.5B" else 8 if fmt == "q4" else 4
        if kind == "step":
            return dict(kind=kind, model=m, layers=layers, fmt=fmt, pos=_log(rng, 8, CONTEXT[m] - 1))
        tokens = _log(rng, 2, 512)
        return dict(kind=kind, model=m, layers=layers, fmt=fmt, tokens=tokens,
                    pos=rng.choice([0, _log(rng, 16, CONTEXT[m] - tokens)]))
    if kind == "turn":
        design, size = rng.choice(["Lusadra", "Girirax"]), rng.choice(["small", "medium", "large"])
        if rng.random() < 0.6:
            return dict(kind=kind, design=design, size=size, prompt=_log(rng, 2, 400), tokens=rng.randint(4, 16))
        return dict(kind=kind, design=design, size=size, prompt=rng.randint(400, 2000), tokens=0)
    if kind == "attention":
        heads, kv_heads, dim = rng.choice([(28, 28, 128), (28, 4, 128), (14, 2, 64), (14, 14, 64)])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=dim, ctx=_log(rng, 100, 32768), kv=rng.choice(["f32", "bf16"]))
    if kind == "product":
        n, k = rng.choice([(4864, 896), (896, 4864), (1152, 896), (3584, 3584), (4608, 3584)])
        return dict(kind=kind, m=_log(rng, 5, 600), n=n + rng.choice([0, 1, -3]), k=k + rng.choice([0, 0, 5]), ta=False,
                    tb=rng.random() < 0.3)
    rows, cols = rng.choice([(4864, 896), (896, 4864), (3584, 3584), (18944, 3584), (3584, 18944)])
    return dict(kind=kind, rows=rows + rng.randint(-40, 40), cols=cols, to=rng.choice(["q4", "bf16"]))


def _config(c):
    """The config.json of a folder design."""
    z = SIZES[c["design"]][c["size"]]
    mlp = {"kind": "dense", "ff": z["ff"]}
    base = {"architecture": c["design"], "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-6}}
    if c["design"] == "Lusadra":
        H, G, D, window = z["left"]
        h, d, v = z["right"]
        left = {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "mask": {"size": window}, "scale": D ** -0.5,
                "q_temp": {"coef": 0.1, "every": 1024}}
        mixer = {"left": left, "right": {"heads": h, "dim": d, "vdim": v, "tau": 16.0}, "left_scale": 0.7, "right_scale": 0.7}
        return dict(base, layers=[{"type": "parallel", "mixer": mixer, "mlp": mlp}] * z["layers"], loop=None)
    h, p, n, g = z["ssm"]
    H, D, R, V, L, Q = z["latent"]
    ssm = {"heads": h, "vdim": p, "state": n, "groups": g, "conv": 4, "norm_groups": g}
    att = {"heads": H, "dim": D, "rot_dim": R, "vdim": V, "kv_rank": L, "q_rank": Q, "scale": (D + R) ** -0.5,
           "rot": {"base": 1e6, "dims": R}}
    pair = [{"type": "mamba2", "mixer": ssm, "mlp": mlp}, {"type": "latent_attention", "mixer": att, "mlp": mlp}]
    return dict(base, embedding={"scale": 4.0}, residual_mult=0.5, layers=pair * (z["layers"] // 2))


# ---- what a program holds before the call -----------------------------------------------------------
class _Closing:
    """A model that is closed with the state that holds it."""

    def __init__(self, m):
        self.m = m

    def __del__(self):
        self.m.close()


class _Buffer:
    """Device memory as the library's calls take it (ptr, nbytes); it lives as long as its tensor."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr, self.nbytes = self.t.data_ptr(), self.t.numel() * self.t.element_size()


def _empty(*shape, dtype=torch.float32):
    return _Buffer(torch.empty(shape, dtype=dtype, device="cuda"))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _tokens(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n)


def _attention_inputs(c, seed):
    g = _generator(seed)
    shape = (c["kv_heads"], c["ctx"], c["dim"])
    q = torch.randn(c["heads"], c["dim"], generator=g, device="cuda")
    k, v = (torch.randn(shape, generator=g, device="cuda") for _ in range(2))
    return q, k.to(_KV[c["kv"]]), v.to(_KV[c["kv"]])


_KV = {"f32": torch.float32, "bf16": torch.bfloat16}


def _product_inputs(c, seed):
    g = _generator(seed)
    a = torch.randn(c["k"] if c["ta"] else c["m"], c["m"] if c["ta"] else c["k"], generator=g, device="cuda")
    b = torch.randn(c["n"] if c["tb"] else c["k"], c["k"] if c["tb"] else c["n"], generator=g, device="cuda") * c["k"] ** -0.5
    return a, b


def _load_input(c, seed):
    return (torch.randn(c["rows"], c["cols"], generator=_generator(seed), device="cuda") * 0.02).to(torch.float16)


def _dims(c):
    return dict(QWEN[c["model"]], n_layers=c["layers"], max_ctx=CONTEXT[c["model"]])


def prepare(case, seed):
    c = case
    lib = pkg.load()
    if c["kind"] in ("step", "prompt"):
        d = _dims(c)
        g = qwen.QwenGPU(d)
        s = dict(case=c, m=_Closing(g))
        g.set_random(seed, c["fmt"])
        g.fill_cache_random(c["pos"], seed)
        s["tokens"] = _tokens(seed, c.get("tokens", 1), d["vocab"])
        return s
    if c["kind"] == "turn":
        z = SIZES[c["design"]][c["size"]]
        m = model.Model.random(_config(c), seed=seed, rank=RANK, max_ctx=4096, chunk=512)
        return dict(case=c, m=_Closing(m), tokens=_tokens(seed, c["prompt"] + c["tokens"], z["vocab"]))
    if c["kind"] == "attention":
        q, k, v = _attention_inputs(c, seed)
        s = dict(case=c, lib=lib, q=_Buffer(q), k=_Buffer(k), v=_Buffer(v), out=_empty(*q.shape))
    elif c["kind"] == "product":
        a, b = _product_inputs(c, seed)
        s = dict(case=c, lib=lib, a=_Buffer(a), b=_Buffer(b), out=_empty(c["m"], c["n"]))
    else:
        n = c["rows"] * c["cols"]
        s = dict(case=c, lib=lib, src=_Buffer(_load_input(c, seed)))
        s["dst"] = _empty(n // 2 + n // 32 * 4, dtype=torch.uint8) if c["to"] == "q4" else _empty(c["rows"], c["cols"], dtype=torch.bfloat16)
    torch.cuda.synchronize()
    return s


def run(state):
    s = state
    c = s["case"]
    if c["kind"] == "step":
        token, logits = s["m"].m.step(int(s["tokens"][0]), c["pos"], want_logits=True)
        return {"token": token, "logits": logits}
    if c["kind"] == "prompt":
        s["m"].m.set_cache_pos(c["pos"])
        return s["m"].m.prefill(s["tokens"])
    if c["kind"] == "turn":
        m, t, n = s["m"].m, s["tokens"], c["prompt"]
        m.reset()
        out = [m.feed(t[:n], [n - 1])]
        for i in range(n, len(t)):
            out.append(m.feed(t[i:i + 1], [0]))
        return out
    lib = s["lib"]
    if c["kind"] == "attention":
        lib.attn_decode(s["q"], s["k"], s["v"], s["out"], c["heads"], c["kv_heads"], c["ctx"], c["ctx"], c["dim"],
                        c["dim"] ** -0.5, kv_bf16=c["kv"] == "bf16")
        return s["out"].t
    if c["kind"] == "product":
        m, n, k = c["m"], c["n"], c["k"]
        lib.gemm(s["a"], m if c["ta"] else k, c["ta"], s["b"], k if c["tb"] else n, c["tb"], s["out"], m, n, k)
        return s["out"].t
    if c["to"] == "q4":
        lib.quantize_q4(s["src"], lib.T_F16, s["dst"], c["rows"], c["cols"])
        packed = c["rows"] * c["cols"] // 2
        return {"packed": s["dst"].t[:packed], "scales": s["dst"].t[packed:].view(torch.float32)}
    lib.convert(s["src"], lib.T_F16, s["dst"], lib.T_BF16, c["rows"] * c["cols"])
    return s["dst"].t


# ---- what a pass cannot do without --------------------------------------------------------------------
def _qwen_weights(d):
    """Weights of a layer and of the head."""
    q, kv = d["n_q_heads"] * d["head_dim"], d["n_kv_heads"] * d["head_dim"]
    return d["hidden"] * (2 * q + 2 * kv + 3 * d["ff"]), d["hidden"] * d["vocab"]


def _turn_weights(c):
    """(weights of all layers, of the head, bytes of state a token reads and writes, numbers per cached position and
    the multiply-adds of a query with one of them, positions a query sees at most), over all layers."""
    z = SIZES[c["design"]][c["size"]]
    n, head = z["layers"], z["width"] * z["vocab"]
    if c["design"] == "Lusadra":
        H, G, D, window = z["left"]
        h, d, v = z["right"]
        layer = z["width"] * (3 * H * D + G * D + 2 * h * d + 3 * h * v + RANK + 2 * z["ff"])
        return n * layer, head, n * 8 * h * d * v, n * 4 * G * D, n * 2 * H * D, window
    h, p, s, g = z["ssm"]
    H, D, R, V, L, Q = z["latent"]
    pair = z["width"] * (3 * h * p + 2 * g * s + h + Q + L + R + 2 * H * V + 6 * z["ff"]) + Q * H * (D + R) + L * H * (D + V)
    return n // 2 * pair, head, n // 2 * 8 * h * p * s, n // 2 * 2 * (L + R), n // 2 * H * (2 * L + R), 1 << 30


def work(case):
    c = case
    if c["kind"] in ("step", "prompt"):
        d, T, per = _dims(c), c.get("tokens", 1), 0.625 if c["fmt"] == "q4" else 2
        layer, head = _qwen_weights(d)
        cached = d["n_layers"] * d["n_kv_heads"] * d["head_dim"] * 2 * 4
        seen = sum(c["pos"] + t + 1 for t in range(T))
        return {"bytes": per * (d["n_layers"] * layer + head) + cached * (c["pos"] + 2 * T) + 4 * d["vocab"],
                "flops": 2 * (d["n_layers"] * layer * T + head) + 4 * d["n_layers"] * d["n_q_heads"] * d["head_dim"] * seen}
    if c["kind"] == "turn":
        layers, head, state, row, query, most = _turn_weights(c)
        P, N, vocab = c["prompt"], c["tokens"], SIZES[c["design"]][c["size"]]["vocab"]
        bytes_ = (2 * (layers + head) + state) * (1 + N) + 4 * vocab * (1 + N)
        bytes_ += row * sum(min(p + 1, most) for p in range(P, P + N)) + row * P
        seen = sum(min(p + 1, most) for p in range(P + N))
        return {"bytes": bytes_, "flops": 2 * (layers * (P + N) + head * (1 + N)) + 2 * query * seen + state * (P + N)}
    if c["kind"] == "attention":
        size = 4 if c["kv"] == "f32" else 2
        return {"bytes": 2 * c["kv_heads"] * c["ctx"] * c["dim"] * size + 8 * c["heads"] * c["dim"],
                "flops": 4 * c["heads"] * c["ctx"] * c["dim"]}
    if c["kind"] == "product":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    return {"bytes": c["rows"] * c["cols"] * (2 + (0.625 if c["to"] == "q4" else 2)), "flops": 0}


def tolerance(case):
    """About four times the distance from 64 bits that was measured over these ranges: f32 sums come out at up to
    3e-7, whole models at up to 1.9e-6, Girirax, whose latents are kept in bf16, at up to 1.1e-3. Bytes stay the same."""
    c = case
    if c["kind"] == "load":
        return "exact"
    if c["kind"] in ("attention", "product"):
        return {"rel": 2e-6}
    return {"rel": 5e-3 if c.get("design") == "Girirax" else 1e-5}


# ---- the same results in 64 bits, from the definitions ---------------------------------------------------
D64 = torch.float64


def _u32(v):
    return v - (1 << 32) if v >= 1 << 31 else v


class _Xorshift:
    """The 32-bit xorshift generator (13, 17, 5) in blocks: a step is linear over GF(2), so a block of 2 m outputs is
    a block of m outputs beside that block moved on by the m-th power of the step."""

    def __init__(self, state):
        self.s = state & 0xffffffff

    @staticmethod
    def _step(x):
        x ^= (x << 13) & 0xffffffff
        x ^= x >> 17
        return x ^ ((x << 5) & 0xffffffff)

    @staticmethod
    def _apply(cols, x):
        y = torch.zeros_like(x)
        for b in range(32):
            y ^= (-((x >> b) & 1)) & _u32(cols[b])
        return y

    def take(self, n):
        """The next n outputs as int32 bits."""
        def one(cols, v):
            y = 0
            for b in range(32):
                if v >> b & 1:
                    y ^= cols[b]
            return y
        x = torch.tensor([_u32(self._step(self.s))], dtype=torch.int32, device="cuda")
        cols = [self._step(1 << b) for b in range(32)]
        while x.numel() < n:
            x = torch.cat([x, self._apply(cols, x[:n - x.numel()])])
            cols = [one(cols, v) for v in cols]
        x = x[:n]
        self.s = int(x[-1]) & 0xffffffff
        return x

    def uniform(self, n):
        """In [-1, 1)."""
        return self.take(n).to(torch.float32) * (1.0 / 2147483648.0)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _tiled(block, n):
    return block.repeat(-(-n // block.numel()))[:n]


def _qwen_exact(c, seed):
    d = _dims(c)
    E, H, G, D, F, T, pos = d["hidden"], d["n_q_heads"], d["n_kv_heads"], d["head_dim"], d["ff"], c.get("tokens", 1), c["pos"]
    r = _Xorshift(seed * 2654435761 + 1)
    words = (32 << 20) // 4
    nib = r.take(words).view(torch.uint8)
    scl = (r.take(words) >> 8 & 0xffffff).to(torch.float32)
    scl = (scl * torch.tensor(0.004, device="cuda")) * (1.0 / 16777216.0) + torch.tensor(0.002, device="cuda")
    bfw = ((r.take(words) & _u32(0x807f807f)) | 0x3c003c00).view(torch.bfloat16)

    def weight(N, K):
        if c["fmt"] == "bf16":
            return _tiled(bfw, N * K).view(N, K)
        p = _tiled(nib, N * K // 2)
        q = torch.stack([p & 15, p >> 4], -1).view(N, K // 32, 32).to(torch.int8) - 8
        return q, _tiled(scl, N * K // 32).view(N, K // 32)

    def times(x, w):
        """x W^T, in row blocks of W."""
        N = len(w) if c["fmt"] == "bf16" else len(w[0])
        out = []
        for i in range(0, N, 16384):
            if c["fmt"] == "bf16":
                m = w[i:i + 16384].to(D64)
            else:
                m = (w[0][i:i + 16384].to(D64) * w[1][i:i + 16384].to(D64)[..., None]).flatten(1)
            out.append(x @ m.T)
        return torch.cat(out, -1)

    def vec(n, mean, std):
        std = torch.tensor(std, dtype=torch.float32, device="cuda")
        return (mean + std * r.uniform(n)).to(D64)

    L = []
    for _ in range(d["n_layers"]):
        L.append([vec(H * D, 0.0, 0.02), vec(G * D, 0.0, 0.02), vec(G * D, 0.0, 0.02), vec(E, 1.0, 0.02), vec(E, 1.0, 0.02)])
    onorm = vec(E, 1.0, 0.02)
    embed = (torch.tensor(0.02, device="cuda") * r.uniform(d["vocab"] * E)).to(torch.bfloat16).view(d["vocab"], E)
    x = embed[torch.from_numpy(_tokens(seed, T, d["vocab"])).cuda()].to(D64)
    del embed
    r = _Xorshift(seed * 2654435761 + 7)
    u = r.uniform(4 * G * d["max_ctx"] * D).view(-1, 4)
    past = (((u[:, 0] + u[:, 1]) + u[:, 2]) + u[:, 3]) * torch.tensor(0.8660254, device="cuda")
    past = past.view(G, d["max_ctx"], D)[:, :pos].to(D64)
    del u
    at = torch.arange(pos, pos + T, device="cuda", dtype=D64)[:, None]
    ang = at * d["rope_base"] ** (-2.0 * torch.arange(D // 2, device="cuda", dtype=D64) / D)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(v):
        a, b = v[..., :D // 2], v[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    mask = torch.ones(T, pos + T, device="cuda", dtype=torch.bool).tril(pos)
    for bq, bk, bv, an, fn in L:
        h = _rms(x, d["eps"]) * an
        qkv = times(h, weight((H + 2 * G) * D, E))
        q = rope((qkv[:, :H * D] + bq).view(T, H, D)).transpose(0, 1)
        k = torch.cat([past, rope((qkv[:, H * D:(H + G) * D] + bk).view(T, G, D)).transpose(0, 1)], 1)
        v = torch.cat([past, (qkv[:, (H + G) * D:] + bv).view(T, G, D).transpose(0, 1)], 1)
        o = torch.empty(T, H * D, dtype=D64, device="cuda")
        for i in range(H):
            s = (q[i] @ k[i // (H // G)].T * D ** -0.5).masked_fill(~mask, -math.inf)
            o[:, i * D:(i + 1) * D] = s.softmax(-1) @ v[i // (H // G)]
        x = x + times(o, weight(E, H * D))
        gu = times(_rms(x, d["eps"]) * fn, weight(2 * F, E))
        x = x + times(_silu(gu[:, :F]) * gu[:, F:], weight(E, F))
    logits = times(_rms(x[-1:], d["eps"]) * onorm, weight(d["vocab"], E))[0]
    return {"token": None, "logits": logits} if c["kind"] == "step" else logits


class _Stream:
    """The seeded weights of a folder design: one block of uniform numbers, walked through again and again."""

    def __init__(self, seed):
        self.block, self.at = _Xorshift(seed * 2654435761 + 1).uniform((1 << 20) + 7), 0

    def __call__(self, rows, cols=0):
        n, B = rows * max(cols, 1), self.block.numel()
        amp = torch.tensor(math.sqrt(np.float32(3.0) / np.float32(cols)) if cols else 1.0, dtype=torch.float32, device="cuda")
        v = (amp * _tiled(self.block.roll(-self.at), n)).to(torch.bfloat16)
        self.at = (self.at + n) % B
        return v.view(rows, cols) if cols else v.to(D64)


def _lin(x, w):
    return torch.cat([x @ w[i:i + 16384].to(D64).T for i in range(0, len(w), 16384)], -1)


def _lusadra_exact(c, z, tokens, seed):
    cfg, S = _config(c), _Stream(seed)
    E, eps, T = z["width"], cfg["norm"]["eps"], len(tokens)
    layers = []
    for lc in cfg["layers"]:
        a, r, ff = lc["mixer"]["left"], lc["mixer"]["right"], lc["mlp"]["ff"]
        hd, rd, rv = a["heads"] * a["dim"], r["heads"] * r["dim"], r["heads"] * r["vdim"]
        w = {"a2": S(rd, RANK), "a2b": S(rd), "rnorm": S(r["vdim"]), "act": S(4), "norm": S(1)}
        for k, n in (("lq", hd), ("lk", a["kv_heads"] * a["dim"]), ("lg", hd), ("rq", rd), ("rk", rd), ("rv", rv), ("rg", rv),
                     ("a1", RANK), ("up", ff)):
            w[k] = S(n, E)
        for k, n in (("lo", hd), ("ro", rv), ("down", ff)):
            w[k] = S(E, n)
        layers.append(w)
    embed, onorm, head = S(z["vocab"], E), S(1), S(z["vocab"], E)
    p = torch.arange(T, device="cuda", dtype=D64)
    col = torch.arange(E, device="cuda")
    ang = p[:, None] * 10000.0 ** (-2.0 * (col // 2).to(D64) / E)
    x = embed[torch.from_numpy(tokens).cuda()].to(D64) + torch.where(col % 2 == 0, ang.sin(), ang.cos())
    for lc, w in zip(cfg["layers"], layers):
        m, a, r = lc["mixer"], lc["mixer"]["left"], lc["mixer"]["right"]
        H, G, D = a["heads"], a["kv_heads"], a["dim"]
        h = _rms(x, eps) * w["norm"]
        temp = 1.0 + a["q_temp"]["coef"] * torch.log(torch.floor((p + 1) / a["q_temp"]["every"]) + 1.0)
        q, k = _lin(h, w["lq"]).view(T, H, D) * temp[:, None, None], _lin(h, w["lk"]).view(T, G, D)
        back = p[:, None] - p[None, :]
        seen = (back >= 0) & (back < a["mask"]["size"])
        o = torch.empty(T, H, D, dtype=D64, device="cuda")
        for i in range(H):
            kk = k[:, i // (H // G)]
            s = q[:, i] @ kk.T * a["scale"] - 2.0 ** (-8.0 * (i + 1) / H) * back
            o[:, i] = s.masked_fill(~seen, -math.inf).softmax(-1) @ kk
        left = _lin(o.flatten(1) * torch.sigmoid(_lin(h, w["lg"])), w["lo"])
        H, D, V = r["heads"], r["dim"], r["vdim"]
        q, k, v = (_lin(h, w[n]).view(T, H, -1) for n in ("rq", "rk", "rv"))
        decay = torch.sigmoid(_lin(_lin(h, w["a1"]), w["a2"]) + w["a2b"]).view(T, H, D) ** (1.0 / r["tau"])
        st, o = torch.zeros(H, D, V, dtype=D64, device="cuda"), torch.empty(T, H, V, dtype=D64, device="cuda")
        for t in range(T):
            st = decay[t, :, :, None] * st + k[t, :, :, None] * v[t, :, None, :]
            o[t] = (q[t, :, :, None] * st).sum(1)
        o = (_rms(o * D ** -0.5, eps) * w["rnorm"]).flatten(1)
        right = _lin(o * _silu(_lin(h, w["rg"])), w["ro"])
        u, (c1, c2, c3, c0) = _lin(h, w["up"]), w["act"]
        y = c1 * _rms(u, eps) + c2 * _rms(u ** 2, eps) + c3 * _rms(u ** 3, eps) + c0
        x = x + m["left_scale"] * left + m["right_scale"] * right + _lin(y, w["down"])
    return _rms(x, eps) * onorm, head


def _girirax_exact(c, z, tokens, seed):
    cfg, S = _config(c), _Stream(seed)
    E, eps, T, mult = z["width"], cfg["norm"]["eps"], len(tokens), cfg["residual_mult"]
    layers = []
    for lc in cfg["layers"]:
        c, ff = lc["mixer"], lc["mlp"]["ff"]
        if lc["type"] == "mamba2":
            inner = c["heads"] * c["vdim"]
            ch = inner + 2 * c["groups"] * c["state"]
            w = {"in": S(inner + ch + c["heads"], E), "conv": S(ch, c["conv"]), "convb": S(ch), "dtb": S(c["heads"]),
                 "A": S(c["heads"]), "D": S(c["heads"]), "mnorm": S(inner)}
        else:
            H = c["heads"]
            inner = H * c["vdim"]
            w = {"dq": S(c["q_rank"], E), "dkv": S(c["kv_rank"] + c["rot_dim"], E), "g": S(inner, E), "dqn": S(c["q_rank"]),
                 "uq": S(H * (c["dim"] + c["rot_dim"]), c["q_rank"]), "kvn": S(c["kv_rank"]), "uk": S(H * c["dim"], c["kv_rank"]),
                 "uv": S(inner, c["kv_rank"])}
        w["o"], w["norm1"] = S(E, inner), S(E)
        w["gate"], w["up"], w["gateb"], w["upb"] = S(ff, E), S(ff, E), S(ff), S(ff)
        w["down"], w["downb"], w["norm2"] = S(E, ff), S(E), S(E)
        layers.append(w)
    onorm, embed = S(E), S(z["vocab"], E)
    p = torch.arange(T, device="cuda", dtype=D64)
    x = embed[torch.from_numpy(tokens).cuda()].to(D64) * cfg["embedding"]["scale"]
    for lc, w in zip(cfg["layers"], layers):
        c = lc["mixer"]
        if lc["type"] == "mamba2":
            H, N, G, V = c["heads"], c["state"], c["groups"], c["vdim"]
            inner, ch = H * V, H * V + 2 * G * N
            u = _lin(x, w["in"])
            gate, xbc, dt = u[:, :inner], u[:, inner:inner + ch], u[:, inner + ch:]
            xbc = torch.cat([torch.zeros(c["conv"] - 1, ch, dtype=D64, device="cuda"), xbc])
            xbc = _silu(sum(w["conv"][:, j].to(D64) * xbc[j:j + T] for j in range(c["conv"])) + w["convb"])
            xs, dt = xbc[:, :inner].view(T, H, V), torch.nn.functional.softplus(dt + w["dtb"], threshold=100.0)
            B, C = (v.view(T, G, N).repeat_interleave(H // G, 1) for v in (xbc[:, inner:inner + G * N], xbc[:, inner + G * N:]))
            keep = torch.exp(-torch.exp(w["A"]) * dt)
            st, y = torch.zeros(H, N, V, dtype=D64, device="cuda"), torch.empty(T, H, V, dtype=D64, device="cuda")
            for t in range(T):
                st = keep[t, :, None, None] * st + (dt[t, :, None] * B[t])[:, :, None] * xs[t, :, None, :]
                y[t] = (C[t, :, :, None] * st).sum(1) + w["D"][:, None] * xs[t]
            y = y.view(T, inner) * _silu(gate)
            y = _rms(y.view(T, c["norm_groups"], -1), eps).flatten(1) * w["mnorm"]
        else:
            H, D, R, V, L = c["heads"], c["dim"], c["rot_dim"], c["vdim"], c["kv_rank"]
            ang = p[:, None] * c["rot"]["base"] ** (-2.0 * torch.arange(R // 2, device="cuda", dtype=D64) / R)

            def turn(v):
                a, b = v[..., :R // 2], v[..., R // 2:]
                cs, sn = (f.view(T, *([1] * (v.dim() - 2)), R // 2) for f in (ang.cos(), ang.sin()))
                return torch.cat([a * cs - b * sn, b * cs + a * sn], -1)

            q = _lin(_rms(_lin(x, w["dq"]), eps) * w["dqn"], w["uq"]).view(T, H, D + R)
            kv = _lin(x, w["dkv"])
            lat, rot = _rms(kv[:, :L], eps) * w["kvn"], turn(kv[:, L:])
            k, v, qr = _lin(lat, w["uk"]).view(T, H, D), _lin(lat, w["uv"]).view(T, H, V), turn(q[..., D:])
            ahead = torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1)
            o = torch.empty(T, H, V, dtype=D64, device="cuda")
            for i in range(H):
                s = (q[:, i, :D] @ k[:, i].T + qr[:, i] @ rot.T) * c["scale"]
                o[:, i] = s.masked_fill(ahead, -math.inf).softmax(-1) @ v[:, i]
            y = o.flatten(1) * torch.sigmoid(_lin(x, w["g"]))
        x = x + mult * _rms(_lin(y, w["o"]), eps) * w["norm1"]
        f = torch.nn.functional.gelu(_lin(x, w["gate"]) + w["gateb"], approximate="tanh") * (_lin(x, w["up"]) + w["upb"])
        x = x + mult * _rms(_lin(f, w["down"]) + w["downb"], eps) * w["norm2"]
    return _rms(x, eps) * onorm, embed


def exact(case, seed):
    c = case
    if c["kind"] in ("step", "prompt"):
        return _qwen_exact(c, seed)
    if c["kind"] == "turn":
        z = SIZES[c["design"]][c["size"]]
        tokens = _tokens(seed, c["prompt"] + c["tokens"], z["vocab"])
        rows, head = (_lusadra_exact if c["design"] == "Lusadra" else _girirax_exact)(c, z, tokens, seed)
        return [v[None] for v in _lin(rows[c["prompt"] - 1:], head)]
    if c["kind"] == "attention":
        q, k, v = _attention_inputs(c, seed)
        rep = c["heads"] // c["kv_heads"]
        out = []
        for h in range(c["heads"]):
            s = (k[h // rep].to(D64) @ q[h].to(D64)) * c["dim"] ** -0.5
            out.append(s.softmax(0) @ v[h // rep].to(D64))
        return torch.stack(out)
    if c["kind"] == "product":
        a, b = _product_inputs(c, seed)
        return (a.T if c["ta"] else a).to(D64) @ (b.T if c["tb"] else b).to(D64)
    w = _load_input(c, seed)
    if c["to"] == "bf16":
        return w.to(D64)
    big = w.to(D64).abs().view(c["rows"], -1, 32).amax(-1)
    return {"packed": None, "scales": big.clamp(min=1e-8).flatten() / 7}
