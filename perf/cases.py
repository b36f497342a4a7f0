"""Performance cases of the quantized linear-layer path.

Each case is one call (or one captured step) that a program using this
framework makes through its public entry points:

* ``dropin``: ``QuantMatrix.matvec`` on NumPy arrays, as an engine that swaps
  the matrix class behind its own model code calls it for every projection;
* ``decode_matrices``: the linear layers of one decode step (RMSNorm, SwiGLU
  and residual adds folded into the launches, and the output head), captured
  once as a HIP graph and replayed per token, as a serving loop runs them;
* ``attention_decode``: rotary embedding, KV store and attention of one token
  over the caches of several layers, captured in the same way;
* ``matmul``: ``matmul_t`` of device-resident rows (M rows of X): small
  batches (a few sequences decoded together, speculative tokens), ragged
  middle sizes, and prompts; every weight format, float32 accuracy by
  default and bf16 / int8 where the caller opts in;
* ``attention_prefill``: causal attention of a prompt chunk;
* ``prefill`` and ``generate``: whole calls of ``Model`` on a 1B-shaped model
  (hidden 2048, 32 query and 8 KV heads, FFN 8192, Q4_K with Q6_K for attn_v,
  some ffn_down and the head) with fewer layers.

Weights are zero-mean blocks of standard deviation about 0.02, activations
N(0, 1), norm weights near one.  Sizes are those of 1B and 8B llama-shaped
models and ragged ones between them.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from alpacca_amd import _lib
from alpacca_amd.model import Hyperparams, Model, Tensor
from alpacca_amd.qmatrix import DenseMatrix, QuantMatrix, matvec_fused_device

DEV = "cuda"
EPS = 1e-5
ROPE_BASE = 500000.0

# values and bytes per block
BLOCK = {"Q4_0": (32, 18), "Q4_1": (32, 20), "Q5_0": (32, 22), "Q5_1": (32, 24),
         "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210),
         "F32": (1, 4), "F16": (1, 2), "BF16": (1, 2)}
DENSE = ("F32", "F16", "BF16")


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # the smallest call: one projection of a 1B-shaped layer on NumPy
        # arrays; latency of the whole host call
        dict(name="dropin_q4k_2048", kind="dropin", dtype="Q4_K", rows=2048, cols=2048),
        # the matrices of an 8B-shaped decode step (two layers and the head):
        # more bytes than the last-level cache, so weights stream from HBM
        dict(name="decode_matrices_8b", kind="decode_matrices", layers=2, hidden=4096,
             kv_dim=1024, ff=14336, vocab=128256),
        # attention of one token late in a 4096-position context, 8B heads
        dict(name="attention_decode_4k", kind="attention_decode", layers=8, n_head=32, n_kv=8,
             head_dim=128, n_ctx=4096, pos=3800),
        # a handful of sequences decoded together
        dict(name="batch_q4k_5", kind="matmul", dtype="Q4_K", rows=14336, cols=4096, m=5,
             precision="auto"),
        # a larger ragged batch in the most common per-32 format
        dict(name="batch_q8_0_27", kind="matmul", dtype="Q8_0", rows=4096, cols=4096, m=27,
             precision="auto"),
        # prompts: the gate/up shape in Q4_K, a ragged prompt through a Q6_K
        # ffn_down
        dict(name="prefill_q4k_512", kind="matmul", dtype="Q4_K", rows=14336, cols=4096, m=512,
             precision="auto"),
        dict(name="prefill_q6k_333", kind="matmul", dtype="Q6_K", rows=4096, cols=14336, m=333,
             precision="auto"),
        # unquantized half-precision weights, an ordinary prompt
        dict(name="prefill_f16_512", kind="matmul", dtype="F16", rows=4096, cols=4096, m=512,
             precision="auto"),
        # the bf16 opt-in
        dict(name="prefill_q4k_bf16_512", kind="matmul", dtype="Q4_K", rows=4096, cols=14336,
             m=512, precision="bf16"),
        # causal attention of a 2048-token prompt, 1B heads
        dict(name="attention_prefill_2k", kind="attention_prefill", n_head=32, n_kv=8,
             head_dim=64, t=2048, pos0=0),
        # a whole batched prefill; a short prompt and its greedy continuation
        dict(name="prefill_1b_2048", kind="prefill", layers=4, vocab=32000, t=2048),
        dict(name="generate_1b", kind="generate", layers=4, vocab=32000, t=200, gen=48),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["dropin", "decode_matrices", "attention_decode", "matmul",
                        "attention_prefill", "prefill", "generate"],
                       weights=[2, 2, 2, 9, 2, 2, 1])[0]
    if kind in ("dropin", "matmul"):
        dtype = rng.choices(["Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "Q4_1", "Q5_0", "Q5_1"],
                            weights=[5, 2, 3, 3, 1, 1, 1, 1])[0]
        if kind == "matmul" and rng.random() < 0.15:
            dtype = rng.choice(DENSE)
        rows = _log_int(rng, 512, 14336)
        step = 256 if BLOCK[dtype][0] == 256 or rng.random() < 0.8 else 32
        cols = step * _log_int(rng, -(-1024 // step), 14336 // step)
        if kind == "dropin":
            return dict(kind=kind, dtype=dtype, rows=rows, cols=cols)
        m = _log_int(rng, 1, 2048)
        while m > 1 and 2.0 * m * rows * cols > 1.2e11:
            m = max(1, m // 2)
        precision = "auto"
        if m >= 64 and rng.random() < 0.25:
            precision = "int8" if dtype == "Q8_0" and rng.random() < 0.5 else "bf16"
        return dict(kind=kind, dtype=dtype, rows=rows, cols=cols, m=m, precision=precision)
    if kind == "decode_matrices":
        hidden = 256 * rng.randint(4, 16)
        return dict(kind=kind, layers=rng.randint(1, 2), hidden=hidden,
                    kv_dim=rng.choice([256, 512, 1024]), ff=256 * rng.randint(8, 56),
                    vocab=_log_int(rng, 8000, 128256))
    if kind == "attention_decode":
        n_kv = rng.choice([4, 8])
        n_ctx = 64 * _log_int(rng, 4, 64)
        return dict(kind=kind, layers=rng.randint(2, 8), n_head=n_kv * rng.choice([1, 2, 4, 8]),
                    n_kv=n_kv, head_dim=rng.choice([64, 128]), n_ctx=n_ctx,
                    pos=rng.randrange(n_ctx))
    if kind == "attention_prefill":
        n_kv = rng.choice([4, 8])
        t = _log_int(rng, 16, 2048)
        return dict(kind=kind, n_head=n_kv * rng.choice([1, 2, 4]), n_kv=n_kv,
                    head_dim=rng.choice([64, 128]), t=t,
                    pos0=rng.choice([0, 0, rng.randrange(1, 1024)]))
    t = _log_int(rng, 20, 2000 if kind == "prefill" else 500)
    case = dict(kind=kind, layers=rng.randint(1, 3), vocab=_log_int(rng, 4000, 32000), t=t)
    if kind == "generate":
        case["gen"] = rng.randint(2, 60)
    return case


# ---- weights -----------------------------------------------------------------

def _gen(seed, k=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1009 + k) % (1 << 62))
    return g


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).view(-1, 2)


def _blocks(dtype, rows, cols, g, std=0.02):
    """The GGUF bytes (uint8, on the GPU) of zero-mean weights."""
    be, bb = BLOCK[dtype]
    if dtype in DENSE:
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[dtype]
        v = torch.randn(rows * cols, generator=g, device=DEV) * std
        return v.to(t).view(torch.uint8)
    nb = rows * (cols // be)
    b = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, generator=g, device=DEV)
    s = std * (0.5 + torch.rand(nb, generator=g, device=DEV))
    if dtype == "Q8_0":
        b[:, 0:2] = _half_bytes(s / 74)
    elif dtype in ("Q4_0", "Q5_0"):
        b[:, 0:2] = _half_bytes(s / (4.6 if dtype == "Q4_0" else 9.2))
    elif dtype in ("Q4_1", "Q5_1"):
        d = s / (4.6 if dtype == "Q4_1" else 9.2)
        b[:, 0:2] = _half_bytes(d)
        b[:, 2:4] = _half_bytes(d * (-7.5 if dtype == "Q4_1" else -15.5))
    elif dtype in ("Q4_K", "Q5_K"):
        # w = d sc q - dmin mn with sc in 32..63, dmin mn close to d sc (codes' mean)
        half = 7.5 if dtype == "Q4_K" else 15.5
        d = (s / (224 if dtype == "Q4_K" else 448)).to(torch.float16).float()
        sc = torch.randint(32, 64, (nb, 8), dtype=torch.int32, generator=g, device=DEV)
        mn = (sc * int(2 * half) + 8) // (16 if dtype == "Q4_K" else 32)
        b[:, 0:2] = _half_bytes(d)
        b[:, 2:4] = _half_bytes(d * (8 if dtype == "Q4_K" else 16))
        b[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
        b[:, 8:12] = (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
        b[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
    else:  # Q6_K
        sc = torch.randint(-32, 32, (nb, 16), dtype=torch.int8, generator=g, device=DEV)
        b[:, 192:208] = sc.view(torch.uint8)
        b[:, 208:210] = _half_bytes(s / 342)
    return b.view(-1)


def _half(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _dense64(dtype, rows, cols, data):
    """The weights as float64, decoded from the GGUF bytes on the GPU."""
    if dtype in DENSE:
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[dtype]
        return data.view(t).to(torch.float64).view(rows, cols)
    be, bb = BLOCK[dtype]
    b = data.view(-1, bb)
    f64 = torch.float64

    def nibbles(q):  # low nibbles, then high ones
        return torch.cat([q & 15, q >> 4], dim=1)

    if dtype == "Q8_0":
        w = b[:, 2:].contiguous().view(torch.int8).to(f64) * _half(b[:, :2])
    elif dtype in ("Q4_0", "Q4_1"):
        q = nibbles(b[:, -16:]).to(f64)
        w = ((q - 8) * _half(b[:, :2]) if dtype == "Q4_0"
             else q * _half(b[:, :2]) + _half(b[:, 2:4]))
    elif dtype in ("Q5_0", "Q5_1"):
        qh = b[:, -20:-16].contiguous().view(torch.int32).to(torch.int64)
        bit = (qh >> torch.arange(32, device=b.device)) & 1
        q = (nibbles(b[:, -16:]).to(torch.int64) | (bit << 4)).to(f64)
        w = ((q - 16) * _half(b[:, :2]) if dtype == "Q5_0"
             else q * _half(b[:, :2]) + _half(b[:, 2:4]))
    elif dtype in ("Q4_K", "Q5_K"):
        s = b[:, 4:16].to(torch.int64)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], dim=1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1)
        qs = b[:, -128:].reshape(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], dim=2).reshape(-1, 8, 32)
        if dtype == "Q5_K":
            bit = (b[:, None, 16:48] >> torch.arange(8, device=b.device,
                                                     dtype=torch.uint8)[:, None]) & 1
            q = q | (bit << 4)
        w = (q.to(f64) * (_half(b[:, 0:2]) * sc)[:, :, None]
             - (_half(b[:, 2:4]) * mn)[:, :, None])
    else:  # Q6_K: 128 low nibbles, 64 high bit pairs, 16 scales, d
        ql, qh = b[:, :128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32)
        lo = torch.cat([ql & 15, ql >> 4], dim=2)
        hi = torch.cat([(qh >> k) & 3 for k in (0, 2, 4, 6)], dim=2)
        q = (lo | (hi << 4)).reshape(-1, 16, 16).to(f64) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(f64)
        w = q * (sc * _half(b[:, 208:210]))[:, :, None]
    return w.reshape(rows, cols)


def _matrix(dtype, rows, cols, data):
    cls = DenseMatrix if dtype in DENSE else QuantMatrix
    return cls(data.cpu().numpy(), dtype, rows, cols)


def _raw_bytes(dtype, rows, cols):
    be, bb = BLOCK[dtype]
    return rows * (cols // be) * bb


# ---- prepare and run -----------------------------------------------------------

def _capture(fn):
    """A HIP graph of fn on a stream of its own, after an eager run of it."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn(s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        fn(s.cuda_stream)
    return g, s


def _layer_shapes(c):
    """Names, formats and shapes of the matrices of layer `i` (Q4_K with Q6_K
    for v and, in every other layer, ffn_down)."""
    h, kv, ff = c["hidden"], c["kv_dim"], c["ff"]
    return lambda i: [("q", "Q4_K", h, h), ("k", "Q4_K", kv, h), ("v", "Q6_K", kv, h),
                      ("o", "Q4_K", h, h), ("gate", "Q4_K", ff, h), ("up", "Q4_K", ff, h),
                      ("down", "Q6_K" if i % 2 else "Q4_K", h, ff)]


def _decode_inputs(c, seed):
    g = _gen(seed, 1)
    h = c["hidden"]
    x = torch.randn(h, generator=g, device=DEV)
    att = torch.randn(c["layers"], h, generator=g, device=DEV)
    norms = 1 + 0.1 * torch.randn(2 * c["layers"] + 1, h, generator=g, device=DEV)
    return x, att, norms


def _prepare_decode(c, seed):
    h, kv, ff = c["hidden"], c["kv_dim"], c["ff"]
    x0, att, norms = _decode_inputs(c, seed)
    layers = []
    for i in range(c["layers"]):
        layers.append({n: _matrix(dt, r, k, _blocks(dt, r, k, _gen(seed, 100 + 10 * i + j)))
                       for j, (n, dt, r, k) in enumerate(_layer_shapes(c)(i))})
    head = _matrix("Q6_K", c["vocab"], h, _blocks("Q6_K", c["vocab"], h, _gen(seed, 99)))
    f32 = dict(dtype=torch.float32, device=DEV)
    x = torch.empty(h, **f32)
    q, k, v = (torch.empty(c["layers"], n, **f32) for n in (h, kv, kv))
    gate, up = torch.empty(ff, **f32), torch.empty(ff, **f32)
    logits = torch.empty(c["vocab"], **f32)

    def step(s):
        x.copy_(x0)
        for i, ly in enumerate(layers):
            n1, n2 = norms[2 * i], norms[2 * i + 1]
            matvec_fused_device([ly["q"], ly["k"], ly["v"]], x.data_ptr(),
                                [q[i].data_ptr(), k[i].data_ptr(), v[i].data_ptr()], s,
                                norm_w_ptr=n1.data_ptr(), eps=EPS, rmsnorm=True)
            matvec_fused_device([ly["o"]], att[i].data_ptr(), [x.data_ptr()], s, accumulate=True)
            matvec_fused_device([ly["gate"], ly["up"]], x.data_ptr(),
                                [gate.data_ptr(), up.data_ptr()], s, norm_w_ptr=n2.data_ptr(),
                                eps=EPS, rmsnorm=True)
            matvec_fused_device([ly["down"]], gate.data_ptr(), [x.data_ptr()], s,
                                x2_ptr=up.data_ptr(), swiglu=True, accumulate=True)
        matvec_fused_device([head], x.data_ptr(), [logits.data_ptr()], s,
                            norm_w_ptr=norms[-1].data_ptr(), eps=EPS, rmsnorm=True)

    graph, stream = _capture(step)
    return dict(graph=graph, out=[q, k, v, x, logits],
                keep=[stream, x0, att, norms, layers, head, gate, up])


def _attn_inputs(c, seed, t, n_ctx, layers=1):
    g = _gen(seed, 2)
    hd, n_kv = c["head_dim"], c["n_kv"]
    q = torch.randn(layers, t, c["n_head"] * hd, generator=g, device=DEV)
    kc = torch.randn(layers, n_kv, n_ctx, hd, generator=g, device=DEV)
    vc = torch.randn(layers, n_kv, n_ctx, hd, generator=g, device=DEV)
    k = torch.randn(layers, n_kv * hd, generator=g, device=DEV)
    v = torch.randn(layers, n_kv * hd, generator=g, device=DEV)
    return q, kc, vc, k, v


def _rope_tables(n_ctx, n_rot):
    """cos / sin of pos * inv_freq in float32: the tables are an input."""
    inv = ROPE_BASE ** (-2.0 * np.arange(n_rot // 2, dtype=np.float32) / n_rot)
    th = np.arange(n_ctx, dtype=np.float32)[:, None] * inv[None, :].astype(np.float32)
    return np.cos(th).astype(np.float32), np.sin(th).astype(np.float32)


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _prepare_attn_decode(c, seed):
    lib = _lib.ensure_device()
    q, kc, vc, k, v = _attn_inputs(c, seed, 1, c["n_ctx"], c["layers"])
    cos, sin = (torch.from_numpy(a).to(DEV) for a in _rope_tables(c["n_ctx"], c["head_dim"]))
    out = torch.empty_like(q)

    def step(s):
        for i in range(c["layers"]):
            _lib.check(lib.aq_attention_rope(
                _p(q[i]), _p(k[i]), _p(v[i]), c["n_head"], c["n_kv"], c["head_dim"],
                c["head_dim"], 0, _p(cos), _p(sin), None, c["pos"], c["n_ctx"], _p(kc[i]),
                _p(vc[i]), _p(out[i]), ctypes.c_void_p(s)))

    graph, stream = _capture(step)
    return dict(graph=graph, out=[out, kc, vc], keep=[stream, q, k, v, cos, sin])


def _model_hp(c):
    return Hyperparams(arch="llama", n_layer=c["layers"], n_embd=2048, n_head=32, n_kv=8,
                       n_ff=8192, n_vocab=c["vocab"], n_ctx_train=4096, head_dim=64, n_rot=64,
                       rms_eps=EPS, rope_base=ROPE_BASE, rope_style="norm")


def _model_weights(c, seed):
    """name -> (dtype, rows, cols, bytes on the GPU), and the norm weights."""
    out, norms, j = {}, {}, 0
    g = _gen(seed, 3)

    def add(name, dtype, rows, cols):
        nonlocal j
        j += 1
        out[name] = (dtype, rows, cols, _blocks(dtype, rows, cols, _gen(seed, 1000 + j)))

    def norm(name):
        norms[name] = 1 + 0.1 * torch.randn(2048, generator=g, device=DEV)

    add("token_embd.weight", "Q4_K", c["vocab"], 2048)
    for i in range(c["layers"]):
        p = f"blk.{i}."
        norm(p + "attn_norm.weight")
        norm(p + "ffn_norm.weight")
        add(p + "attn_q.weight", "Q4_K", 2048, 2048)
        add(p + "attn_k.weight", "Q4_K", 512, 2048)
        add(p + "attn_v.weight", "Q6_K", 512, 2048)
        add(p + "attn_output.weight", "Q4_K", 2048, 2048)
        add(p + "ffn_gate.weight", "Q4_K", 8192, 2048)
        add(p + "ffn_up.weight", "Q4_K", 8192, 2048)
        add(p + "ffn_down.weight", "Q6_K" if i % 2 else "Q4_K", 2048, 8192)
    norm("output_norm.weight")
    add("output.weight", "Q6_K", c["vocab"], 2048)
    return out, norms


def _tokens(c, seed):
    rng = np.random.default_rng(seed + 17)
    return [int(t) for t in rng.integers(0, c["vocab"], c["t"])]


def _prepare_model(c, seed):
    weights, norms = _model_weights(c, seed)
    tensors = {n: Tensor(dt, (r, k), b.cpu().numpy()) for n, (dt, r, k, b) in weights.items()}
    for n, v in norms.items():
        tensors[n] = Tensor("F32", (2048,), v.cpu().numpy())
    n_ctx = c["t"] if c["kind"] == "prefill" else 1024
    return dict(model=Model(_model_hp(c), tensors, n_ctx=n_ctx), tokens=_tokens(c, seed),
                gen=c.get("gen", 0))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode_matrices":
        st = _prepare_decode(case, seed)
    elif kind == "attention_decode":
        st = _prepare_attn_decode(case, seed)
    elif kind in ("prefill", "generate"):
        st = _prepare_model(case, seed)
    elif kind == "attention_prefill":
        t, p0 = case["t"], case["pos0"]
        q, kc, vc, _k, _v = _attn_inputs(case, seed, t, p0 + t)
        _lib.ensure_device()
        st = dict(q=q, kc=kc, vc=vc, out=torch.empty_like(q), case=case)
    else:
        dt, r, k = case["dtype"], case["rows"], case["cols"]
        W = _matrix(dt, r, k, _blocks(dt, r, k, _gen(seed, 4)))
        g = _gen(seed, 5)
        X = torch.randn(case.get("m", 1), k, generator=g, device=DEV)
        if kind == "dropin":
            st = dict(W=W, x=X[0].cpu().numpy())
        else:
            st = dict(W=W, X=X, precision=None if case["precision"] == "auto"
                      else case["precision"])
    torch.cuda.synchronize()
    st["kind"] = kind
    return st


def run(state):
    kind = state["kind"]
    if kind == "dropin":
        return state["W"].matvec(state["x"])
    if kind == "matmul":
        return state["W"].matmul_t(state["X"], precision=state["precision"])
    if kind in ("decode_matrices", "attention_decode"):
        state["graph"].replay()
        return state["out"]
    if kind == "attention_prefill":
        c = state["case"]
        _lib.check(_lib.load().aq_attention_batch(
            _p(state["q"]), _p(state["kc"]), _p(state["vc"]), c["t"], c["n_head"], c["n_kv"],
            c["head_dim"], c["pos0"] + c["t"], None, c["pos0"], _p(state["out"]),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        return state["out"]
    model = state["model"]
    if kind == "prefill":
        model.reset()
        return [model.prefill(state["tokens"]), model.kv]
    tokens = model.generate_greedy(state["tokens"], state["gen"])
    return [np.asarray(tokens, dtype=np.int64), model.logits]


# ---- work and tolerance ----------------------------------------------------------

def _model_work(c, tokens, heads, ctx_pairs):
    """Bytes and flops of `tokens` tokens through the layers in one pass over
    the weights, `heads` heads, `ctx_pairs` (query, position) pairs."""
    per = [("Q4_K", 2048, 2048), ("Q4_K", 512, 2048), ("Q6_K", 512, 2048),
           ("Q4_K", 2048, 2048), ("Q4_K", 16384, 2048)]
    wb = fl = 0
    for i in range(c["layers"]):
        for dt, r, k in per + [("Q6_K" if i % 2 else "Q4_K", 2048, 8192)]:
            wb += _raw_bytes(dt, r, k)
            fl += 2 * r * k * tokens
    wb += _raw_bytes("Q6_K", c["vocab"], 2048)
    fl += 2 * c["vocab"] * 2048 * heads
    fl += c["layers"] * ctx_pairs * 2048 * 4
    return wb, fl


def work(case):
    c, kind = case, case["kind"]
    if kind in ("dropin", "matmul"):
        m = c.get("m", 1)
        return {"bytes": _raw_bytes(c["dtype"], c["rows"], c["cols"])
                + 4 * m * (c["rows"] + c["cols"]),
                "flops": 2 * m * c["rows"] * c["cols"]}
    if kind == "decode_matrices":
        ms = [s for i in range(c["layers"]) for s in _layer_shapes(c)(i)]
        ms.append(("head", "Q6_K", c["vocab"], c["hidden"]))
        return {"bytes": sum(_raw_bytes(dt, r, k) + 4 * r for _n, dt, r, k in ms),
                "flops": sum(2 * r * k for _n, _dt, r, k in ms)}
    if kind == "attention_decode":
        n = c["pos"] + 1
        return {"bytes": c["layers"] * 4 * c["head_dim"] * (2 * n * c["n_kv"] + 2 * c["n_head"]),
                "flops": c["layers"] * 4 * c["n_head"] * c["head_dim"] * n}
    if kind == "attention_prefill":
        t, p0, hd = c["t"], c["pos0"], c["head_dim"]
        return {"bytes": 4 * hd * (2 * t * c["n_head"] + 2 * (t + p0) * c["n_kv"]),
                "flops": 4 * c["n_head"] * hd * (t * p0 + t * (t + 1) // 2)}
    t = c["t"]
    wb, fl = _model_work(c, t, 1, t * (t + 1) // 2)
    kv = c["layers"] * 2 * 512 * 4
    if kind == "prefill":
        return {"bytes": wb + kv * t + _raw_bytes("Q4_K", t, 2048) + 4 * c["vocab"], "flops": fl}
    steps = c["gen"] - 1
    mean = t + steps // 2
    swb, sfl = _model_work(c, steps, steps, steps * mean)
    return {"bytes": wb + kv * t + steps * (swb + kv * mean), "flops": fl + sfl}


def tolerance(case):
    """About four times the error measured against exact() (in brackets)."""
    kind = case["kind"]
    if kind == "matmul" and case["precision"] == "bf16":
        return {"rel": 1e-2}  # X and W rounded to bf16 (2.4e-3)
    if kind == "matmul" and case["precision"] == "int8":
        return {"rel": 2.5e-2}  # X rounded to int8 per 32 values (5.4e-3)
    if kind in ("matmul", "dropin"):
        # codes and mins of Q4_1 / Q5_1 cancel in zero-mean weights (6e-6;
        # the other formats up to 8e-7)
        return {"rel": 2.5e-5 if case["dtype"] in ("Q4_1", "Q5_1") else 3e-6}
    if kind == "decode_matrices":
        return {"rel": 1e-5}  # (2.3e-6)
    if kind in ("prefill", "generate"):
        return {"rel": 1.5e-5, "differ": 0.0}  # (2.7e-6)
    return {"rel": 2e-6}  # attention (4e-7)


# ---- the same outputs in 64 bits ---------------------------------------------------

def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(torch.float64)


def _silu64(g):
    return g / (1 + torch.exp(-g))


def _rope64(x, cos, sin):
    """Adjacent pairs of x [t, heads, hd] rotated by the rows of the tables."""
    x0, x1 = x[..., 0::2], x[..., 1::2]
    c, s = cos[:, None, :], sin[:, None, :]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], dim=-1).flatten(-2)


def _attend64(q, kc, vc, p0):
    """q [t, n_head, hd] at positions p0.. over kc, vc [n_kv, >= p0 + t, hd]."""
    t, n_head, hd = q.shape
    g = n_head // kc.shape[0]
    out = torch.empty_like(q)
    n = p0 + t
    mask = torch.arange(n, device=q.device)[None, :] > (p0 + torch.arange(t, device=q.device))[:, None]
    for h in range(n_head):
        s = (q[:, h] @ kc[h // g, :n].T) / math.sqrt(hd)
        s.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(s, dim=-1) @ vc[h // g, :n]
    return out


class _Model64:
    def __init__(self, c, seed):
        weights, norms = _model_weights(c, seed)
        self.w = {n: _dense64(dt, r, k, b) for n, (dt, r, k, b) in weights.items()}
        self.norms = norms
        self.c = c
        n_ctx = c["t"] + c.get("gen", 0)
        cos, sin = _rope_tables(n_ctx, 64)
        self.cos, self.sin = (torch.from_numpy(a).to(DEV, torch.float64) for a in (cos, sin))
        self.kv = torch.zeros(c["layers"], 2, 8, n_ctx, 64, dtype=torch.float64, device=DEV)
        self.n = 0

    def step(self, tokens):
        w, n, t = self.w, self.n, len(tokens)
        x = w["token_embd.weight"][torch.tensor(tokens, device=DEV)]
        cos, sin = self.cos[n:n + t], self.sin[n:n + t]
        for i in range(self.c["layers"]):
            p = f"blk.{i}."
            h = _rms64(x, self.norms[p + "attn_norm.weight"])
            q = _rope64((h @ w[p + "attn_q.weight"].T).view(t, 32, 64), cos, sin)
            k = _rope64((h @ w[p + "attn_k.weight"].T).view(t, 8, 64), cos, sin)
            self.kv[i, 0, :, n:n + t] = k.transpose(0, 1)
            self.kv[i, 1, :, n:n + t] = (h @ w[p + "attn_v.weight"].T).view(t, 8, 64).transpose(0, 1)
            a = _attend64(q, self.kv[i, 0], self.kv[i, 1], n).reshape(t, 2048)
            x = x + a @ w[p + "attn_output.weight"].T
            h = _rms64(x, self.norms[p + "ffn_norm.weight"])
            act = _silu64(h @ w[p + "ffn_gate.weight"].T) * (h @ w[p + "ffn_up.weight"].T)
            x = x + act @ w[p + "ffn_down.weight"].T
        self.n += t
        return _rms64(x[-1], self.norms["output_norm.weight"]) @ w["output.weight"].T


def exact(case, seed):
    c, kind = case, case["kind"]
    f64 = torch.float64
    if kind in ("dropin", "matmul"):
        dt, r, k = c["dtype"], c["rows"], c["cols"]
        W = _dense64(dt, r, k, _blocks(dt, r, k, _gen(seed, 4)))
        X = torch.randn(c.get("m", 1), k, generator=_gen(seed, 5), device=DEV)
        Y = X.to(f64) @ W.T
        return Y[0].cpu().numpy() if kind == "dropin" else Y
    if kind == "decode_matrices":
        x0, att, norms = _decode_inputs(c, seed)
        x = x0.to(f64)
        outs = [[], [], []]
        for i in range(c["layers"]):
            W = {n: _dense64(dt, r, k, _blocks(dt, r, k, _gen(seed, 100 + 10 * i + j)))
                 for j, (n, dt, r, k) in enumerate(_layer_shapes(c)(i))}
            h = _rms64(x, norms[2 * i])
            for o, n in zip(outs, "qkv"):
                o.append(W[n] @ h)
            x = x + W["o"] @ att[i].to(f64)
            h = _rms64(x, norms[2 * i + 1])
            x = x + W["down"] @ (_silu64(W["gate"] @ h) * (W["up"] @ h))
        head = _dense64("Q6_K", c["vocab"], c["hidden"],
                        _blocks("Q6_K", c["vocab"], c["hidden"], _gen(seed, 99)))
        return [torch.stack(o) for o in outs] + [x, head @ _rms64(x, norms[-1])]
    if kind == "attention_decode":
        q, kc, vc, k, v = (t.to(f64) for t in _attn_inputs(c, seed, 1, c["n_ctx"], c["layers"]))
        hd, n_kv, p = c["head_dim"], c["n_kv"], c["pos"]
        cos, sin = (torch.from_numpy(a[p:p + 1]).to(DEV, f64)
                    for a in _rope_tables(c["n_ctx"], hd))
        out = torch.empty_like(q)
        for i in range(c["layers"]):
            kc[i, :, p] = _rope64(k[i].view(1, n_kv, hd), cos, sin)[0]
            vc[i, :, p] = v[i].view(n_kv, hd)
            qr = _rope64(q[i].view(1, c["n_head"], hd), cos, sin)
            out[i] = _attend64(qr, kc[i], vc[i], p).reshape(1, -1)
        return [out, kc, vc]
    if kind == "attention_prefill":
        t, p0 = c["t"], c["pos0"]
        q, kc, vc, _k, _v = _attn_inputs(c, seed, t, p0 + t)
        o = _attend64(q[0].view(t, c["n_head"], c["head_dim"]).to(f64), kc[0].to(f64),
                      vc[0].to(f64), p0)
        return o.reshape(1, t, -1)
    model = _Model64(c, seed)
    logits = model.step(_tokens(c, seed))
    if kind == "prefill":
        return [logits.cpu().numpy(), model.kv]
    out = [int(torch.argmax(logits))]
    for _ in range(c["gen"] - 1):
        logits = model.step([out[-1]])
        out.append(int(torch.argmax(logits)))
    return [np.asarray(out, dtype=np.int64), logits]
