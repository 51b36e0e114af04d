"""What the performance of this backend is measured on: the work a program that
uses it has it do, through the public entry points, from one row of a decode
step to a whole request.

  linear   Context.qlinear / qlinear_swiglu: a block-quantized projection of
           M activation rows (1: decode, 2..16: several sequences decoded
           together, more: prompt rows).
  attend   KVCache.attention_decode: one token's attention over a filled cache.
  sdp      Context.sdp_attention: the engine's per-op attention over f32 K/V.
  mlp      layer_norm, gemm_f32, gelu, gemm_f32, add: the engine's per-op calls
           of a GELU feed-forward block, f32.
  layers   Model.forward_hidden: prompt rows through decoder layers, in chunks.
  request  Model.prefill_mfma, generate_ids, step: a prompt, a greedy run and
           the logits of the token after it.

Everything is drawn from the seed: activations of unit scale, N(0, 0.02)
weights quantized to the blocks the library takes, norm weights near 1.
"""
import math
import zlib

import numpy as np
import torch

import vlrf_amd as V

DTYPES = {"q8_0": V.DT_Q8_0, "q4_0": V.DT_Q4_0, "f32": V.DT_F32}
KV = {"q8_0": V.KV_Q8_0, "f16": V.KV_F16, "f32": V.KV_F32}
EPS, THETA = 1e-5, 10000.0

# The decoder shapes of the benchmarks (vlrf_amd/formats.py: llama_1b, llama8b_layer, tiny).
SHAPES = {
    "1.1B": dict(d_model=2048, d_ff=5632, n_heads=32, n_kv_heads=4),
    "8B": dict(d_model=4096, d_ff=14336, n_heads=32, n_kv_heads=8),
    "tiny": dict(d_model=256, d_ff=704, n_heads=4, n_kv_heads=1),
}


def listed():
    return [
        # The down projection of a decode step at the 1.1B shape, called on its own: the smallest call.
        dict(name="down_1b_1_row", op="linear", N=2048, K=5632, M=1, dtype="q8_0", swiglu=False, norm=False,
             residual=True),
        # Gate and up with SwiGLU for six sequences decoded together.
        dict(name="gate_up_1b_6_rows", op="linear", N=5632, K=2048, M=6, dtype="q8_0", swiglu=True, norm=True,
             residual=False),
        # The fused QKV projection of a short prompt or a batch of sequences, at the 8B shape.
        dict(name="qkv_8b_100_rows", op="linear", N=6144, K=4096, M=100, dtype="q4_0", swiglu=False, norm=True,
             residual=False),
        # The down projection of a long prompt at the 8B shape.
        dict(name="down_8b_1777_rows", op="linear", N=4096, K=14336, M=1777, dtype="q8_0", swiglu=False, norm=False,
             residual=True),
        # Decode attention over the quantized cache at the length of the attention benchmark.
        dict(name="attend_1b_4096_q8", op="attend", H=32, G=4, d=64, ctx=4096, kv="q8_0"),
        # The same of a long conversation at the 8B shape over an f16 cache.
        dict(name="attend_8b_15001_f16", op="attend", H=32, G=8, d=128, ctx=15001, kv="f16"),
        # Causal attention of a prompt through the engine's per-op interface.
        dict(name="sdp_777_causal", op="sdp", H=32, d=64, T=777, ctx=777, causal=True),
        # A feed-forward block of the engine's per-op interface for a prompt.
        dict(name="mlp_f32_300", op="mlp", T=300, D=768, F=3072),
        # Prompt rows through one layer of the 8B shape: the prefill benchmark's length.
        dict(name="layer_8b_2048", op="layers", shape="8B", L=1, T=2048, chunks=1, dtype="q8_0", kv="q8_0"),
        # A prompt that arrives in chunks, each attending to the chunks before it.
        dict(name="layers_1b_3_chunks", op="layers", shape="1.1B", L=2, T=700, chunks=3, dtype="q4_0", kv="f16"),
        # A request to the 1.1B model of the decode benchmark: a long prompt, then a greedy run.
        dict(name="request_1b_2000_48", op="request", shape="1.1B", L=22, vocab=32000, prompt=2000, gen=48,
             dtype="q8_0", kv="q8_0"),
        # A short request at the 8B shape (four layers, as the 8B decode benchmark), 4-bit weights.
        dict(name="request_8b_90_24", op="request", shape="8B", L=4, vocab=32000, prompt=90, gen=24, dtype="q4_0",
             kv="q8_0"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["linear", "linear", "linear", "attend", "attend", "sdp", "mlp", "layers", "request"])
    if op == "linear":
        M = _log(rng, 1, 2048)
        dtype = rng.choice(["q8_0", "q8_0", "q4_0", "q4_0", "f32"] if M <= 16 else ["q8_0", "q4_0"])
        N, K = _log(rng, 256, 14336), 64 * _log(rng, 4, 224)
        swiglu = rng.random() < 0.3
        return dict(op=op, N=N, K=K, M=M, dtype=dtype, swiglu=swiglu, norm=rng.random() < 0.5,
                    residual=not swiglu and rng.random() < 0.5)
    if op == "attend":
        H, G, d = rng.choice([(32, 4, 64), (32, 8, 128), (8, 8, 64), (16, 8, 64), (8, 2, 128)])
        return dict(op=op, H=H, G=G, d=d, ctx=_log(rng, 48, 16384), kv=rng.choice(["q8_0", "q8_0", "f16", "f32"]))
    if op == "sdp":
        T = _log(rng, 1, 1024)
        return dict(op=op, H=rng.choice([8, 12, 32]), d=rng.choice([64, 64, 80, 128]), T=T,
                    ctx=T + rng.choice([0, 0, _log(rng, 1, 1024)]), causal=rng.random() < 0.7)
    if op == "mlp":
        D = 64 * _log(rng, 4, 25)
        return dict(op=op, T=_log(rng, 1, 1024), D=D, F=4 * D)
    dtype, kv = rng.choice(["q8_0", "q4_0"]), rng.choice(["q8_0", "q8_0", "f16", "f32"])
    if op == "layers":
        shape, L = rng.choice([("8B", 1), ("1.1B", 2), ("1.1B", 4), ("tiny", 2)])
        T = _log(rng, 32, 2048)
        return dict(op=op, shape=shape, L=L, T=T, chunks=rng.choice([1, 1, min(3, T)]), dtype=dtype, kv=kv)
    shape, L = rng.choice([("8B", 2), ("1.1B", 8), ("tiny", 2)])
    return dict(op=op, shape=shape, L=L, vocab=rng.choice([32000, 32000, 5003]), prompt=_log(rng, 8, 2000),
                gen=_log(rng, 4, 48), dtype=dtype, kv=kv)


# ---- inputs ------------------------------------------------------------------
_CTX = []


def _context():
    if not _CTX:                       # one context for the program, as a server keeps it
        _CTX.append(V.Context(0))
    return _CTX[0]


class Buf:
    """A torch tensor as the binding takes buffers: its device address and size."""

    def __init__(self, t):
        assert t.is_contiguous() and t.is_cuda
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _normal(seed, name, shape, std=1.0):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFFFFFF)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std)


def _norm_weight(seed, name, D):
    return 1.0 + _normal(seed, name, (D,), 0.1)


def _quantized(w, dtype):
    """(host payload, decode) of f32 rows w [N, K]: the blocks the library uploads
    (Q8_0: f16 scale amax/127 and 32 codes; Q4_0: f16 scale of the signed
    extreme over -8 and 16 bytes, element 2j in the low nibble of byte j), and
    the f64 values they stand for."""
    N, K = w.shape
    if dtype == "f32":
        return w.cpu().numpy(), lambda: w.double()
    b = w.view(N, K // 32, 32)
    if dtype == "q8_0":
        d = (b.abs().amax(-1, keepdim=True) / 127.0).half()
        q = (b / d.float()).round_().clamp_(-127, 127).to(torch.int8)
        codes, values = q.view(torch.uint8), q
    else:
        at = b.abs().argmax(-1, keepdim=True)
        d = (b.gather(-1, at) / -8.0).half()
        q = (b / d.float() + 8.5).to(torch.int32).clamp_(0, 15).to(torch.uint8)
        codes, values = q[..., 0::2] | (q[..., 1::2] << 4), q.to(torch.int8) - 8
    payload = torch.cat([d.view(torch.uint8), codes], -1).view(N, -1).cpu().numpy()
    return payload, lambda: (values.double() * d.double()).view(N, K)


def _linear_inputs(c, seed):
    N, K, M = c["N"], c["K"], c["M"]
    ws = [_quantized(_normal(seed, f"w{i}", (N, K), 0.02), c["dtype"]) for i in range(2 if c["swiglu"] else 1)]
    x = _normal(seed, "x", (M, K))
    nw = _norm_weight(seed, "norm", K) if c["norm"] else None
    res = _normal(seed, "residual", (M, N)) if c["residual"] else None
    return ws, x, nw, res


def _attend_inputs(c, seed):
    row = c["G"] * c["d"]
    # queries of twice the unit scale: scores of a standard deviation of two
    return (_normal(seed, "q", (c["H"], c["d"]), 2.0), _normal(seed, "k", (c["ctx"], row)),
            _normal(seed, "v", (c["ctx"], row)))


def _sdp_inputs(c, seed):
    return (_normal(seed, "q", (c["H"], c["T"], c["d"]), 2.0), _normal(seed, "k", (c["H"], c["ctx"], c["d"])),
            _normal(seed, "v", (c["H"], c["ctx"], c["d"])))


def _mlp_inputs(c, seed):
    T, D, F = c["T"], c["D"], c["F"]
    return (_normal(seed, "x", (T, D)), _norm_weight(seed, "ln.w", D), _normal(seed, "ln.b", (D,), 0.1),
            _normal(seed, "w1", (F, D), 0.02), _normal(seed, "w2", (D, F), 0.02))


def _config(c):
    cfg = dict(SHAPES[c["shape"]], n_layers=c["L"], norm_eps=EPS, rope_theta=THETA, weight_dtype=DTYPES[c["dtype"]],
               kv_dtype=KV[c["kv"]])
    if c["op"] == "layers":            # the rows come embedded: a small vocabulary, as the prefill benchmark
        return dict(cfg, vocab_size=256, max_seq_len=c["T"])
    return dict(cfg, vocab_size=c["vocab"], max_seq_len=c["prompt"] + c["gen"] + 8)


def _layer_tensors(cfg, seed, l):
    """(name, f32 [rows, cols]) of layer l, one at a time."""
    D, F = cfg["d_model"], cfg["d_ff"]
    dkv = cfg["n_kv_heads"] * (D // cfg["n_heads"])
    for name in ("ln1", "ln2"):
        yield f"layers.{l}.{name}.weight", _norm_weight(seed, f"{l}.{name}", D).view(1, D)
    for name, n, k in (("attn.q_proj", D, D), ("attn.k_proj", dkv, D), ("attn.v_proj", dkv, D),
                       ("attn.o_proj", D, D), ("ffn.gate", F, D), ("ffn.fc1", F, D), ("ffn.fc2", D, F)):
        yield f"layers.{l}.{name}.weight", _normal(seed, f"{l}.{name}", (n, k), 0.02)


def _head_tensors(cfg, seed):
    """The embedding, the final norm and the LM head.  Row j of the head holds
    the direction of token follow(j)'s embedding: as in a trained model, the
    greedy token wins by a wide margin, while every logit carries the whole
    computation."""
    W, D = cfg["vocab_size"], cfg["d_model"]
    embed = _normal(seed, "embed", (W, D))
    follow = (torch.arange(W, device="cuda") * 7919 + 13 + int(seed) % 1000) % W
    yield "embed.weight", embed
    yield "ln_final.weight", _norm_weight(seed, "ln_final", D).view(1, D)
    yield "lm_head.weight", embed[follow] * 0.02


def _prompt(c, seed):
    return np.random.default_rng([int(seed), 77]).integers(0, c["vocab"], c["prompt"], dtype=np.int32)


def _model(c, seed):
    cfg = _config(c)
    m = V.Model(_context(), cfg)
    groups = [_head_tensors(cfg, seed)] + [_layer_tensors(cfg, seed, l) for l in range(cfg["n_layers"])]
    for group in groups:
        for name, w in group:
            f32 = "ln" in name or "embed" in name
            payload, _ = _quantized(w, "f32" if f32 else c["dtype"])
            m.set_weight(name, payload, V.DT_F32 if f32 else DTYPES[c["dtype"]], *w.shape)
    return m


def _chunks(c):
    at = [c["T"] * i // c["chunks"] for i in range(c["chunks"] + 1)]
    return [(a, b) for a, b in zip(at, at[1:]) if b > a]


def prepare(case, seed):
    c, ctx, op = case, _context(), case["op"]
    if op == "linear":
        ws, x, nw, res = _linear_inputs(c, seed)
        s = dict(w=[V.QuantWeight(ctx, p, DTYPES[c["dtype"]], c["N"], c["K"]) for p, _ in ws], x=Buf(x),
                 y=Buf(torch.empty(c["M"], c["N"], device="cuda")), norm=Buf(nw) if nw is not None else None,
                 residual=Buf(res) if res is not None else None)
    elif op == "attend":
        q, k, v = _attend_inputs(c, seed)
        kv = V.KVCache(ctx, 1, c["ctx"], c["G"], c["d"], KV[c["kv"]])
        torch.cuda.synchronize()
        kv.append(0, Buf(k), Buf(v), c["ctx"])
        ctx.sync()
        s = dict(kv=kv, q=Buf(q), out=Buf(torch.empty(c["H"], c["d"], device="cuda")))
    elif op == "sdp":
        q, k, v = _sdp_inputs(c, seed)
        s = dict(q=Buf(q), k=Buf(k), v=Buf(v), out=Buf(torch.empty_like(q)))
    elif op == "mlp":
        x, w, b, w1, w2 = _mlp_inputs(c, seed)
        s = dict(x=Buf(x), w=Buf(w), b=Buf(b), w1=Buf(w1), w2=Buf(w2), n=Buf(torch.empty_like(x)),
                 h=Buf(torch.empty(c["T"], c["F"], device="cuda")), y=Buf(torch.empty_like(x)))
    elif op == "layers":
        x = _normal(seed, "x", (c["T"], SHAPES[c["shape"]]["d_model"]))
        out = torch.empty_like(x)
        s = dict(m=_model(c, seed), out=out, parts=[(Buf(x[a:b]), Buf(out[a:b])) for a, b in _chunks(c)])
    else:
        s = dict(m=_model(c, seed), prompt=_prompt(c, seed))
    torch.cuda.synchronize()           # torch's stream made the inputs; the context has its own
    return dict(s, case=c, ctx=ctx)


def run(state):
    s, c, ctx = state, state["case"], state["ctx"]
    op = c["op"]
    if op == "linear":
        if c["swiglu"]:
            ctx.qlinear_swiglu(s["w"][0], s["w"][1], s["x"], s["y"], c["M"], s["norm"], EPS)
        else:
            ctx.qlinear(s["w"][0], s["x"], s["y"], c["M"], s["norm"], EPS, s["residual"])
        return s["y"].t
    if op == "attend":
        s["kv"].attention_decode(0, s["q"], s["out"], c["H"], c["ctx"], 1.0 / math.sqrt(c["d"]))
        return s["out"].t
    if op == "sdp":
        ctx.sdp_attention(s["q"], s["k"], s["v"], s["out"], c["H"], c["T"], c["ctx"], c["d"],
                          1.0 / math.sqrt(c["d"]), c["causal"])
        return s["out"].t
    if op == "mlp":
        T, D, F = c["T"], c["D"], c["F"]
        ctx.layer_norm(s["x"], s["w"], s["b"], s["n"], T, D, EPS)
        ctx.gemm_f32(s["n"], s["w1"], s["h"], T, F, D, trans_b=True)
        ctx.gelu(s["h"], T * F)
        ctx.gemm_f32(s["h"], s["w2"], s["y"], T, D, F, trans_b=True)
        ctx.add(s["y"], s["x"], T * D)
        return s["y"].t
    m = s["m"]
    m.reset()                          # a new request
    if op == "layers":
        for x, out in s["parts"]:
            m.forward_hidden(x, out)
        return s["out"]
    first = m.prefill_mfma(s["prompt"])
    ids = m.generate_ids(first, c["gen"])
    last, logits = m.step(int(ids[-1]), want_logits=True)
    return dict(first=first, ids=ids, last=last, logits=logits)


# ---- what a pass cannot do without ---------------------------------------------
def _wbytes(dtype, n):
    return n * {"q8_0": 34 / 32, "q4_0": 18 / 32, "f32": 4}[dtype]


def _kvbytes(kv, rows, row):
    """K and V rows of a cache, with the row scales of the quantized one."""
    return 2 * rows * (row * {"q8_0": 1, "f16": 2, "f32": 4}[kv] + (4 if kv == "q8_0" else 0))


def work(case):
    c, op = case, case["op"]
    if op == "linear":
        n = 2 if c["swiglu"] else 1
        rows = c["M"] * (c["K"] + c["N"] * (2 if c["residual"] else 1)) + (c["K"] if c["norm"] else 0)
        return dict(bytes=n * _wbytes(c["dtype"], c["N"] * c["K"]) + 4 * rows, flops=2 * n * c["M"] * c["N"] * c["K"])
    if op == "attend":
        return dict(bytes=_kvbytes(c["kv"], c["ctx"], c["G"] * c["d"]) + 8 * c["H"] * c["d"],
                    flops=4 * c["H"] * c["d"] * c["ctx"])
    if op == "sdp":
        T, n = c["T"], c["ctx"]
        pairs = T * (n - T) + T * (T + 1) // 2 if c["causal"] else T * n
        return dict(bytes=8 * c["H"] * c["d"] * (T + n), flops=4 * c["H"] * c["d"] * pairs)
    if op == "mlp":
        T, D, F = c["T"], c["D"], c["F"]
        return dict(bytes=4 * (2 * T * D + 2 * D + 2 * D * F), flops=4 * T * D * F)
    cfg = _config(c)
    D, F, L, H = cfg["d_model"], cfg["d_ff"], cfg["n_layers"], cfg["n_heads"]
    dkv = cfg["n_kv_heads"] * (D // H)
    per = D * (2 * D + 2 * dkv) + 3 * D * F                     # weights of a layer
    if op == "layers":
        T = c["T"]
        return dict(bytes=L * (_wbytes(c["dtype"], per) * len(_chunks(c)) + _kvbytes(c["kv"], T, dkv)) + 8 * T * D,
                    flops=L * (2 * T * per + 2 * T * (T + 1) * D))
    T, n, W = c["prompt"], c["gen"] + 1, c["vocab"]             # decode steps, each over all weights and its context
    ctx = sum(T + 1 + i for i in range(n))
    return dict(bytes=(n + 1) * (L * _wbytes(c["dtype"], per) + _wbytes(c["dtype"], W * D)) +
                L * _kvbytes(c["kv"], T + ctx, dkv) + 4 * D * (T + n) + 4 * W,
                flops=L * (2 * T * per + 2 * T * (T + 1) * D) + 2 * n * (L * per + W * D) + 4 * L * D * ctx)


def tolerance(case):
    """About four times the largest distance from exact() over the ranges of draw()."""
    c, op = case, case["op"]
    if op == "linear":
        # f32 products of one row 2e-7; up to 16 rows as two bf16 halves of x 4e-6; above, both
        # operands rounded to bf16, 2e-3 (the product of two of them in SwiGLU 3.5e-3)
        return {"rel": 1e-6} if c["M"] == 1 else {"rel": 1.5e-5} if c["M"] <= 16 else {"rel": 1e-2}
    if op in ("attend", "sdp", "mlp"):
        return {"rel": 4e-6}                                    # f32 throughout: up to 1e-6
    return {"rel": 2e-2} if op == "layers" else {"rel": 3e-2}   # bf16 operands in every layer: 6e-3, logits 1.2e-2


# ---- the same in 64 bits -------------------------------------------------------
def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _cached(x, kv):
    """f64 rows as the cache of this type gives them back."""
    x = x.float()
    if kv == "f32":
        return x.double()
    if kv == "f16":                    # mantissa rounded half up, values below the normal range flushed
        y = ((x.contiguous().view(torch.int32) + 0x1000) & ~0x1FFF).view(torch.float32)
        return torch.where(y.abs() < 2.0 ** -14, torch.zeros_like(y), y).double()
    # each step in 64 bits and rounded once: torch divides by a constant in 32 bits by its reciprocal
    s = (x.abs().amax(-1, keepdim=True).double() / 127.0).float().double()
    y = (x.double() * (1.0 / s).float().double()).float()
    q = torch.trunc(y + torch.where(y < 0, -0.5, 0.5)).clamp_(-127, 127)
    return q.double() * s


def _attention64(q, k, v, scale, first):
    """q [H, T, d] over k, v [H, ctx, d]; query i sees keys up to first + i (all when first is None)."""
    H, T, _ = q.shape
    out = torch.empty_like(q)
    for h in range(H):
        p = (q[h] @ k[h].t()).mul_(scale)
        if first is not None:
            keys = torch.arange(k.shape[1], device=q.device)
            p.masked_fill_(keys[None, :] > first + torch.arange(T, device=q.device)[:, None], float("-inf"))
        out[h] = torch.softmax(p, -1) @ v[h]
    return out


class _Decoder64:
    def __init__(self, c, seed):
        self.c, self.seed, self.cfg = c, seed, _config(c)
        cfg = self.cfg
        self.dh = cfg["d_model"] // cfg["n_heads"]
        self.layers = [self._decoded(_layer_tensors(cfg, seed, l)) for l in range(cfg["n_layers"])]
        self.cache = [None] * cfg["n_layers"]
        half = self.dh // 2
        freq = np.float32(1) / np.power(np.float32(THETA), np.arange(0, self.dh, 2, dtype=np.float32) /
                                        np.float32(self.dh), dtype=np.float32)
        angle = (np.arange(cfg["max_seq_len"], dtype=np.float32)[:, None] * freq[None, :half]).astype(np.float64)
        self.cos = torch.from_numpy(np.cos(angle)).cuda()[:, None, :]
        self.sin = torch.from_numpy(np.sin(angle)).cuda()[:, None, :]

    def _decoded(self, tensors):
        """f64 for a few layers; a whole model is held in f32 (which holds code times scale) and widened when used."""
        got = {}
        for name, w in tensors:
            f32 = "ln" in name or "embed" in name
            got[name.split(".", 2)[-1] if name.startswith("layers") else name] = _quantized(
                w, "f32" if f32 else self.c["dtype"])[1]().float()
        return got

    def _rope(self, x, pos):
        half = self.dh // 2
        c, s = self.cos[pos:pos + x.shape[0]], self.sin[pos:pos + x.shape[0]]
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    def forward(self, x, pos):
        cfg, T = self.cfg, x.shape[0]
        H, G, d = cfg["n_heads"], cfg["n_kv_heads"], self.dh
        for l, w in enumerate(self.layers):
            h = _rms64(x, w["ln1.weight"].double())
            q = self._rope((h @ w["attn.q_proj.weight"].double().t()).view(T, H, d), pos)
            k = self._rope((h @ w["attn.k_proj.weight"].double().t()).view(T, G, d), pos).reshape(T, G * d)
            v = h @ w["attn.v_proj.weight"].double().t()
            new = torch.stack([_cached(k, self.c["kv"]), _cached(v, self.c["kv"])])
            kv = new if pos == 0 else torch.cat([self.cache[l], new], 1)
            self.cache[l] = kv
            rows = kv.view(2, pos + T, G, d).transpose(1, 2).repeat_interleave(H // G, 1)
            att = _attention64(q.transpose(0, 1), rows[0], rows[1], 1.0 / math.sqrt(d), pos)
            x = x + att.transpose(0, 1).reshape(T, H * d) @ w["attn.o_proj.weight"].double().t()
            h = _rms64(x, w["ln2.weight"].double())
            g = h @ w["ffn.gate.weight"].double().t()
            h = g * torch.sigmoid(g) * (h @ w["ffn.fc1.weight"].double().t())
            x = x + h @ w["ffn.fc2.weight"].double().t()
        return x


def exact(case, seed):
    c, op = case, case["op"]
    if op == "linear":
        ws, x, nw, res = _linear_inputs(c, seed)
        x = x.double()
        if nw is not None:
            x = _rms64(x, nw.double())
        y = x @ ws[0][1]().t()
        if c["swiglu"]:
            y = y * torch.sigmoid(y) * (x @ ws[1][1]().t())
        return y if res is None else y + res.double()
    if op == "attend":
        q, k, v = _attend_inputs(c, seed)
        H, G, d = c["H"], c["G"], c["d"]
        k, v = (_cached(t, c["kv"]).view(c["ctx"], G, d).transpose(0, 1).repeat_interleave(H // G, 0) for t in (k, v))
        return _attention64(q.double().view(H, 1, d), k, v, 1.0 / math.sqrt(d), None).view(H, d)
    if op == "sdp":
        q, k, v = (t.double() for t in _sdp_inputs(c, seed))
        return _attention64(q, k, v, 1.0 / math.sqrt(c["d"]), c["ctx"] - c["T"] if c["causal"] else None)
    if op == "mlp":
        x, w, b, w1, w2 = (t.double() for t in _mlp_inputs(c, seed))
        h = torch.nn.functional.layer_norm(x, (c["D"],), w, b, EPS) @ w1.t()
        return x + torch.nn.functional.gelu(h, approximate="tanh") @ w2.t()
    m = _Decoder64(c, seed)
    if op == "layers":
        x = _normal(seed, "x", (c["T"], m.cfg["d_model"])).double()
        return torch.cat([m.forward(x[a:b], a) for a, b in _chunks(c)])
    head = m._decoded(_head_tensors(m.cfg, seed))

    def logits(tokens, pos):
        x = m.forward(head["embed.weight"][torch.as_tensor(tokens, device="cuda").long()].double(), pos)
        return _rms64(x[-1:], head["ln_final.weight"].double()) @ head["lm_head.weight"].double().t()

    first = int(logits(_prompt(c, seed), 0).argmax())
    ids, pos = [], c["prompt"]
    for i in range(c["gen"]):
        ids.append(int(logits([ids[-1] if ids else first], pos + i).argmax()))
    end = logits([ids[-1]], pos + c["gen"])[0]
    return dict(first=first, ids=np.array(ids, np.int32), last=int(end.argmax()), logits=end)
