"""Performance cases: the work a user of this backend has it do.

A case is one call through `flarellm_amd.backend` on inputs that a program
already holds.  The kinds:

  decode     one token through a model with a filled KV cache, logits on the
             host (`HipBackend.forward_single_token_gpu`)
  verify     a speculative batch of drafts through a model in one pass
             (`HipBackend.verify`)
  prefill    a prompt through a model from an empty cache, logits of its last
             token (`HipBackend.forward_prefill`)
  project    one quantized projection of a batch of rows
             (`HipBackend.batched_dequant_matmul`)
  matvec     one quantized projection of one row, already quantized
             (`HipBackend.matvec_q8in`)
  logits     the output projection of 1..8 f32 rows
             (`HipBackend.batched_matvec_f32in` / `matvec_f32in`)
  kvattn     decode attention of one query over a filled cache
             (`HipBackend.grouped_query_attention_from_gpu_cache`)
  selfattn   causal attention of a whole prompt, f32 rows
             (`HipBackend.prefill_attention_gpu`)

Shapes are those of `flarellm_amd.synth` (SmolLM2-135M, Llama-3.2-1B and
Llama-3-8B) and sizes between them.  Weights are N(0, 0.02) rows quantized to
the GGUF formats, activations N(0, 1), norms N(1, 0.1); cached keys and
values N(0, 1), which is what such weights make of a normalized row.
"""
import math

import numpy as np
import torch

from flarellm_amd import FL_KV_F16, FL_KV_F32, FL_KV_KIVI2, FL_KV_Q8, FL_Q4K, FL_Q6K, FL_Q8_0
from flarellm_amd.backend import HipBackend
from flarellm_amd.synth import ModelSpec, QWeight, SynthModel

FORMATS = {"q8_0": FL_Q8_0, "q4_k": FL_Q4K, "q6_k": FL_Q6K}
CACHES = {"f32": FL_KV_F32, "f16": FL_KV_F16, "q8": FL_KV_Q8, "kivi2": FL_KV_KIVI2}
EPS = 1e-5
# Weights of a model repeat after this many layers (each layer is still its
# own tensor on the device): a checkpoint is read from a file, and making
# billions of random weights here would only cost time.
DISTINCT_LAYERS = 2


def _model(kind, hidden, layers, heads, kv_heads, head_dim, inter, vocab, fmt, embed, output, theta, **more):
    return dict(kind=kind, hidden=hidden, layers=layers, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                inter=inter, vocab=vocab, fmt=fmt, embed=embed, output=output, theta=theta, **more)


def _smol_135m(kind, **more):
    return _model(kind, 576, 30, 9, 3, 64, 1536, 49152, "q8_0", "q8_0", "", 100000.0, **more)


def _llama_1b(kind, layers, **more):
    return _model(kind, 2048, layers, 32, 8, 64, 8192, 128256, "q8_0", "q8_0", "", 500000.0, **more)


def _llama_8b(kind, layers, **more):
    return _model(kind, 4096, layers, 32, 8, 128, 14336, 128256, "q4_k", "q6_k", "q6_k", 500000.0, **more)


def listed():
    return [
        # smallest: one projection of a SmolLM2-135M layer, launch and wait
        dict(name="matvec_576x1536_q8_0", kind="matvec", fmt="q8_0", rows=576, cols=1536),
        # a chat turn on the smallest model: every kernel is latency
        _smol_135m("decode", name="decode_135m", cache="f16", context=100),
        # four layers and the head of the benchmark's decode workload, its
        # context half way through (few layers: see tolerance)
        _llama_1b("decode", 4, name="decode_1b_layers", cache="f16", context=640),
        # layers and head of the 8B shape at a long context
        _llama_8b("decode", 2, name="decode_8b_layers", cache="f16", context=4100),
        # a speculative step: eight drafts behind a long context
        _llama_8b("verify", 2, name="verify_8b_layers", cache="f16", context=4096, tokens=8),
        # time to first token of an ordinary prompt (odd length)
        _llama_1b("prefill", 4, name="prefill_1b_layers_509", cache="f16", context=0, tokens=509),
        # time to first token of a long document on the 8B shape
        _llama_8b("prefill", 2, name="prefill_8b_layers_4096", cache="f16", context=0, tokens=4096),
        # the gate projection of a prompt, layer by layer (ComputeBackend)
        dict(name="project_q4_k_1000", kind="project", fmt="q4_k", rows=14336, cols=4096, batch=1000),
        # a down projection of a short, odd batch
        dict(name="project_q8_0_77", kind="project", fmt="q8_0", rows=2048, cols=8192, batch=77),
        # the output projection of a speculative batch, full logits
        dict(name="logits_q6_k_8", kind="logits", fmt="q6_k", rows=128256, cols=4096, batch=8),
        # decode attention at the longest context, 2-bit cache
        dict(name="kvattn_kivi2_128k", kind="kvattn", cache="kivi2", heads=32, kv_heads=8, head_dim=128,
             context=131072),
        # a prompt's attention, layer by layer (ComputeBackend), odd length
        dict(name="selfattn_1531", kind="selfattn", heads=32, kv_heads=8, head_dim=128, tokens=1531),
    ]


def draw(rng):
    def spread(lo, hi, step=1):  # spread over the logarithm, both ends in
        v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return min(hi, max(lo, v // step * step))

    kind = rng.choice(["decode", "verify", "prefill", "prefill", "project", "project", "matvec", "logits", "kvattn",
                       "selfattn"])
    if kind in ("decode", "verify", "prefill"):
        head_dim = rng.choice([64, 128])
        kv_heads, group = rng.choice([(2, 4), (3, 3), (4, 2), (4, 8), (8, 4), (8, 4), (8, 1)])
        fmt = rng.choice(["q8_0", "q4_k"])
        if fmt == "q4_k" and kv_heads * group * head_dim % 256:
            fmt = "q8_0"
        step = 256 if fmt == "q4_k" else 64
        embed = "q8_0" if fmt == "q8_0" else "q6_k"
        c = _model(kind, spread(512, 4096, step), rng.randint(1, 2), kv_heads * group, kv_heads, head_dim,
                   spread(1024, 14336, step), spread(8000, 64000), fmt, embed, embed if fmt == "q4_k" else "",
                   rng.choice([10000.0, 500000.0]), cache=rng.choice(["f16", "f16", "f16", "q8"]), context=0)
        if kind == "prefill":
            c["cache"] = rng.choice(["f16", "f16", "f16", "f16", "q8", "f32"])
            c["tokens"] = spread(2, 2500)
        else:
            c["context"] = spread(16, 8000)
        if kind == "verify":
            c["tokens"] = rng.choice([2, 3, 4, 5, 6, 8])
        return c
    if kind in ("project", "matvec"):
        fmt = rng.choice(["q8_0", "q4_k"])
        c = dict(kind=kind, fmt=fmt, rows=spread(192, 16384), cols=spread(512, 14336, 256 if fmt == "q4_k" else 32))
        if kind == "project":
            c["batch"] = spread(2, 2000)
        return c
    if kind == "logits":
        return dict(kind=kind, fmt=rng.choice(["q6_k", "q8_0"]), rows=spread(16000, 128256),
                    cols=spread(512, 4096, 256), batch=rng.choice([1, 2, 3, 5, 8]))
    head_dim = rng.choice([64, 128])
    kv_heads, group = rng.choice([(2, 4), (3, 3), (4, 8), (8, 4), (8, 2)])
    c = dict(kind=kind, heads=kv_heads * group, kv_heads=kv_heads, head_dim=head_dim)
    if kind == "kvattn":
        c.update(cache=rng.choice(["f16", "q8", "kivi2"]), context=spread(64, 100000))
    else:
        c["tokens"] = spread(16, 2000)
    return c


# ---- inputs -------------------------------------------------------------------


class _Source:
    """Normal values on the GPU from (seed, stream)."""

    def __init__(self, seed):
        self.seed, self.stream = int(seed), 0

    def normal(self, *shape, mean=0.0, std=1.0):
        self.stream += 1
        g = torch.Generator(device="cuda").manual_seed(self.seed * 1000003 + self.stream)
        return torch.randn(*shape, device="cuda", generator=g).mul_(std).add_(mean)

    def tokens(self, n, vocab):
        self.stream += 1
        return np.random.default_rng([self.seed, self.stream]).integers(0, vocab, n, dtype=np.uint32)


def _half_bytes(h):
    return h.half().view(torch.uint8).view(-1, 2)


def _encode(w, fmt):
    """GGUF blocks of the rows of w: (bytes [rows, row bytes], the values that
    the blocks stand for as 64-bit floats)."""
    rows, cols = w.shape
    if fmt == "q8_0":
        b = w.view(-1, 32)
        d = (b.abs().amax(1, keepdim=True) / 127.0).half()
        q = torch.clamp(torch.round(b / d.float()), -127, 127)
        q = torch.where(d > 0, q, torch.zeros_like(q)).to(torch.int8)
        raw = torch.cat([_half_bytes(d), q.view(torch.uint8)], 1)
        return raw.view(rows, -1), lambda: (q.double() * d.double()).view(rows, cols)
    if fmt == "q4_k":
        b = w.view(-1, 8, 32)
        lo = b.amin(2).clamp(max=0.0)
        scale, least = (b.amax(2) - lo) / 15.0, -lo
        d = (scale.amax(1, keepdim=True) / 63.0).half()
        dmin = (least.amax(1, keepdim=True) / 63.0).half()
        sc = torch.clamp(torch.round(scale / d.float()), 0, 63)
        mn = torch.clamp(torch.round(least / dmin.float()), 0, 63)
        q = torch.round((b + (dmin.float() * mn)[..., None]) / (d.float() * sc).clamp(min=1e-12)[..., None])
        q = torch.clamp(q, 0, 15).to(torch.uint8)
        s, m = sc.to(torch.uint8), mn.to(torch.uint8)
        head = torch.cat([_half_bytes(d), _half_bytes(dmin), s[:, :4] | ((s[:, 4:] & 3) << 6),
                          m[:, :4] | ((m[:, 4:] & 3) << 6), (s[:, 4:] >> 2) | ((m[:, 4:] >> 2) << 4)], 1)
        raw = torch.cat([head, (q[:, :4] | (q[:, 4:] << 4)).reshape(-1, 128)], 1)
        return raw.view(rows, -1), lambda: (q.double() * (d.double() * sc.double())[..., None]
                                            - (dmin.double() * mn.double())[..., None]).view(rows, cols)
    b = w.view(-1, 16, 16)  # q6_k
    top = b.gather(2, b.abs().argmax(2, keepdim=True)).squeeze(2)
    scale = -top / 32.0
    d = (-scale.gather(1, scale.abs().argmax(1, keepdim=True)) / 128.0).half()
    sc = torch.clamp(torch.round(scale / d.float()), -128, 127)
    q = torch.clamp(torch.round(b / (d.float() * sc)[..., None]), -32, 31).to(torch.int8)
    u = (q + 32).to(torch.uint8).view(-1, 2, 4, 32)  # [block, half, quarter, value]
    ql = (u[:, :, :2] & 15) | ((u[:, :, 2:] & 15) << 4)
    qh = (u >> 4)[:, :, 0] | ((u >> 4)[:, :, 1] << 2) | ((u >> 4)[:, :, 2] << 4) | ((u >> 4)[:, :, 3] << 6)
    raw = torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _half_bytes(d)], 1)
    return raw.view(rows, -1), lambda: (q.double() * (d.double() * sc.double())[..., None]).view(rows, cols)


def _weight(src, rows, cols, fmt, exact=False):
    """A quantized N(0, 0.02) weight: its GGUF bytes on the host, or with
    exact the values in 64 bits on the GPU."""
    raw, values = _encode(src.normal(rows, cols, std=0.02), fmt)
    return values() if exact else QWeight(raw.cpu().numpy().reshape(-1), FORMATS[fmt], rows, cols)


def _spec(c):
    room = c["context"] + c.get("tokens", 1)
    return ModelSpec("case", c["hidden"], c["layers"], c["heads"], c["kv_heads"], c["head_dim"], c["inter"],
                     c["vocab"], (room + 127) // 64 * 64, FORMATS[c["fmt"]], FORMATS[c["embed"]],
                     FORMATS[c["output"]] if c["output"] else None, EPS, c["theta"])


def _model_inputs(c, seed, exact=False):
    """(layers, attention norms, FFN norms, output norm, embedding, cached rows
    per layer, tokens) in the order the seed makes them."""
    src, spec = _Source(seed), _spec(c)
    layers, attn, ffn = [], [], []
    for _ in range(min(DISTINCT_LAYERS, c["layers"])):
        layers.append([_weight(src, r, k, c["fmt"], exact) for r, k in spec.layer_shapes()])
        attn.append(src.normal(c["hidden"], mean=1.0, std=0.1))
        ffn.append(src.normal(c["hidden"], mean=1.0, std=0.1))
    last = src.normal(c["hidden"], mean=1.0, std=0.1)
    embedding = _weight(src, c["vocab"], c["hidden"], c["embed"], exact)
    kvd = c["kv_heads"] * c["head_dim"]
    rows = [(src.normal(c["context"], kvd), src.normal(c["context"], kvd))
            for _ in range(min(DISTINCT_LAYERS, c["layers"]))] if c["context"] else []
    return layers, attn, ffn, last, embedding, rows, src.tokens(c.get("tokens", 1), c["vocab"])


def _prepare_model(c, seed):
    layers, attn, ffn, last, embedding, rows, tokens = _model_inputs(c, seed)
    spec, n = _spec(c), len(layers)
    model = SynthModel(spec)
    for i in range(spec.layers):
        model.layers.append(layers[i % n])
        model.attn_norms.append(attn[i % n].cpu().numpy())
        model.ffn_norms.append(ffn[i % n].cpu().numpy())
    model.output_norm = last.cpu().numpy()
    model.embedding = embedding
    model.output = embedding if c["output"] else None  # same bytes, a tensor of its own
    backend = HipBackend(0)
    backend.init_gpu_kv_cache(spec, CACHES[c["cache"]])
    backend.upload_weights_to_gpu(model)
    host = [(k.cpu().numpy(), v.cpu().numpy()) for k, v in rows]
    for i in range(spec.layers if host else 0):
        backend.gpu_kv_write_batch(i, 0, *host[i % n])
    return dict(backend=backend, kind=c["kind"], tokens=tokens, position=c["context"])


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("decode", "verify", "prefill"):
        return _prepare_model(c, seed)
    src, backend = _Source(seed), HipBackend(0)
    state = dict(backend=backend, kind=kind)
    if kind in ("project", "matvec", "logits"):
        state["weight"] = backend.upload(_weight(src, c["rows"], c["cols"], c["fmt"]))
        x = src.normal(c.get("batch", 1), c["cols"])
        if kind == "matvec":
            state["x"] = backend.quantize_q8(x[0])
        else:
            state["x"] = x[0] if kind == "logits" and c["batch"] == 1 else x
    elif kind == "kvattn":
        spec = ModelSpec("case", 256, 1, c["heads"], c["kv_heads"], c["head_dim"], 256, 256,
                         (c["context"] + 63) // 64 * 64, FL_Q8_0, FL_Q8_0, None)
        backend.init_gpu_kv_cache(spec, CACHES[c["cache"]])
        kvd = c["kv_heads"] * c["head_dim"]
        k, v = src.normal(c["context"], kvd), src.normal(c["context"], kvd)
        backend.gpu_kv_write_batch(0, 0, k.cpu().numpy(), v.cpu().numpy())
        state["q"] = src.normal(c["heads"] * c["head_dim"]).cpu().numpy()
        state["context"] = c["context"]
    else:
        kvd = c["kv_heads"] * c["head_dim"]
        state["qkv"] = tuple(src.normal(c["tokens"], n) for n in (c["heads"] * c["head_dim"], kvd, kvd))
        state["shape"] = (c["tokens"], c["heads"], c["kv_heads"], c["head_dim"])
    return state


def run(state):
    b, kind = state["backend"], state["kind"]
    if kind == "decode":
        return b.forward_single_token_gpu(int(state["tokens"][0]), state["position"])
    if kind == "verify":
        # the winning logit of every draft; the token ids beside them may
        # differ where two logits of a random model tie
        return b.verify(state["tokens"], state["position"])[1]
    if kind == "prefill":
        return b.forward_prefill(state["tokens"], 0)[0]
    if kind == "project":
        return b.batched_dequant_matmul(state["weight"], state["x"])
    if kind == "matvec":
        return b.matvec_q8in(state["weight"], *state["x"])
    if kind == "logits":
        x = state["x"]
        return b.matvec_f32in(state["weight"], x) if x.dim() == 1 else b.batched_matvec_f32in(state["weight"], x)
    if kind == "kvattn":
        return b.grouped_query_attention_from_gpu_cache(state["q"], 0, state["context"])
    return b.prefill_attention_gpu(*state["qkv"], *state["shape"])


# ---- what a pass cannot do without ---------------------------------------------

ROW_BITS = {"q8_0": 34 * 8 / 32, "q4_k": 144 * 8 / 256, "q6_k": 210 * 8 / 256}  # per weight


def _cache_bytes(cache, values):
    """K and V of `values` cached values each."""
    per = {"f32": 4.0, "f16": 2.0, "q8": 1 + 2 / 32, "kivi2": 0.25 + 4 / 32}[cache]
    return 2 * values * per


def work(case):
    c, kind = case, case["kind"]
    if kind in ("project", "matvec", "logits"):
        m, n, k = c.get("batch", 1), c["rows"], c["cols"]
        each = k * (1 + 8 / 32) if kind == "matvec" else 4.0 * k
        return dict(bytes=n * k * ROW_BITS[c["fmt"]] / 8 + m * (each + 4.0 * n), flops=2.0 * m * n * k)
    if kind in ("kvattn", "selfattn"):
        qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        if kind == "kvattn":
            return dict(bytes=_cache_bytes(c["cache"], c["context"] * kvd) + 8.0 * qd, flops=4.0 * c["context"] * qd)
        t = c["tokens"]
        return dict(bytes=8.0 * t * (qd + kvd), flops=2.0 * t * (t + 1) * qd)
    n, past = c.get("tokens", 1), c["context"]
    qd, kvd, h, f = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["hidden"], c["inter"]
    weights = c["layers"] * (h * (qd + 2 * kvd) + qd * h + 3 * h * f)
    head = c["vocab"] * h
    heads = n if kind == "verify" else 1  # tokens whose logits are formed
    pairs = n * past + n * (n + 1) / 2
    return dict(bytes=weights * ROW_BITS[c["fmt"]] / 8 + head * ROW_BITS[c["output"] or c["embed"]] / 8
                + c["layers"] * _cache_bytes(c["cache"], (past + n) * kvd)
                + (0 if kind == "verify" else 4.0 * c["vocab"]),
                flops=2.0 * n * weights + 2.0 * heads * head + c["layers"] * 4.0 * pairs * qd)


def tolerance(case):
    if case["kind"] in ("decode", "verify", "prefill"):
        # Every projection requantizes its input to 8 bits, so a last-bit
        # difference of one sum moves a code by a step.  Measured between a
        # prompt in one pass and the same tokens one at a time, and between
        # either and 64 bits: 0.007 after one layer, 0.016 after two and 0.020
        # after four of these shapes (0.0035 for the 30 layers of the smallest
        # model), at most 0.12 of the root mean square.
        return {"rel": 0.03, "max": 0.4}
    # f32 sums of exact products: 1e-7 to 4e-7 against 64 bits, 1e-6 to 2e-6
    # for the largest difference; 2e-6 where the 2-bit cache's minima cancel
    # in the mean over a long context
    return {"rel": 8e-6, "max": 8e-5} if case.get("cache") == "kivi2" else {"rel": 2e-6, "max": 2e-5}


# ---- the same in 64 bits ---------------------------------------------------------


def _over(a, b):
    """a / b rounded once (by a number, torch multiplies by a reciprocal)."""
    a, b = (v if torch.is_tensor(v) else torch.full_like(w, v) for v, w in ((a, b), (b, a)))
    return a / b


def _rounded(y):
    """Halves away from zero, exact for a float y."""
    return torch.sign(y) * torch.floor(y.double().abs() + 0.5).to(y.dtype)


def _quantized(x):
    """Rows as the backend's 8-bit activations: per 32 values a scale
    max/127 and codes rounded half away from zero, in the type of x."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    top = b.abs().amax(-1, keepdim=True)
    y = b * torch.where(top > 0, _over(127.0, top), torch.zeros_like(top))
    return (_rounded(y).double() * _over(top, 127.0).double()).view(x.shape)


def _cached(k, v, cache, kv_heads, head_dim):
    """Cached rows as the cache form stores them, in 64 bits."""
    if cache == "f32":
        return k.double(), v.double()
    if cache == "q8":
        def one(x):
            b = x.float().reshape(x.shape[0], -1, 32)
            top = b.abs().amax(-1, keepdim=True)
            y = b * torch.where(top > 0, _over(127.0, top), torch.zeros_like(top))
            return (_rounded(y) * _over(top, 127.0).half().float()).view(x.shape).double()
        return one(k), one(v)
    k, v = k.float().half().float(), v.float().half().float()
    if cache == "kivi2":
        t = k.shape[0]
        old = 32 * ((t - 129) // 32) if t > 129 else 0

        def one(g):  # [..., 32]
            lo = g.amin(-1, keepdim=True)
            span = g.amax(-1, keepdim=True) - lo
            code = torch.clamp(_rounded((g - lo) * _over(3.0, span)), 0, 3)
            return code * _over(span, 3.0).half().float() + lo.half().float()

        if old:
            k[:old] = one(k[:old].view(-1, 32, k.shape[1]).transpose(1, 2)).transpose(1, 2).reshape(old, -1)
            v[:old] = one(v[:old].reshape(old, -1, 32)).reshape(old, -1)
    return k.double(), v.double()


def _attend(q, k, v, heads, kv_heads, head_dim):
    """Causal attention of the last len(q) rows of the cache, 64 bits."""
    n, t = q.shape[0], k.shape[0]
    q = q.view(n, kv_heads, heads // kv_heads, head_dim)
    k, v = k.view(t, kv_heads, head_dim), v.view(t, kv_heads, head_dim)
    seen = torch.arange(t, device=q.device)[None, :] <= torch.arange(t - n, t, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(kv_heads):
        for g in range(heads // kv_heads):
            s = q[:, h, g] @ k[:, h].T / math.sqrt(head_dim)
            out[:, h, g] = torch.softmax(s.masked_fill(~seen, -math.inf), 1) @ v[:, h]
    return out.view(n, -1)


def _exact_model(c, seed):
    layers, attn, ffn, last, embedding, rows, tokens = _model_inputs(c, seed, exact=True)
    n, past, half = len(tokens), c["context"], c["head_dim"] // 2
    position = np.arange(past, past + n, dtype=np.float32)
    rate = np.float32(1) / np.power(np.float32(c["theta"]), np.float32(2) * np.arange(half, dtype=np.float32)
                                    / np.float32(c["head_dim"]))
    angle = torch.from_numpy(position[:, None] * rate[None, :]).cuda().double()[:, None, :]
    cos, sin = torch.cos(angle), torch.sin(angle)

    def turned(y):
        y = y.view(n, -1, 2 * half)
        a, b = y[..., :half], y[..., half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1).reshape(n, -1)

    def norm(y, w):
        return y / torch.sqrt(y.square().mean(1, keepdim=True) + EPS) * w.double()

    x = embedding[torch.from_numpy(tokens.astype(np.int64)).cuda()].clone()
    shape = (c["heads"], c["kv_heads"], c["head_dim"])
    for i in range(c["layers"]):
        wq, wk, wv, wo, gate, up, down = layers[i % len(layers)]
        y = _quantized(norm(x, attn[i % len(layers)]))
        k, v = turned(y @ wk.T), y @ wv.T
        if past:
            k, v = (torch.cat([a.double(), b]) for a, b in zip(rows[i % len(layers)], (k, v)))
        k, v = _cached(k, v, c["cache"], *shape[1:])
        x = x + _quantized(_attend(turned(y @ wq.T), k, v, *shape)) @ wo.T
        y = _quantized(norm(x, ffn[i % len(layers)]))
        g = y @ gate.T
        x = x + _quantized(g / (1 + torch.exp(-g)) * (y @ up.T)) @ down.T
    x = norm(x if c["kind"] == "verify" else x[-1:], last)
    logits = x @ embedding.T
    return logits.amax(1) if c["kind"] == "verify" else logits[0]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("decode", "verify", "prefill"):
        return _exact_model(c, seed)
    src = _Source(seed)
    if kind in ("project", "matvec", "logits"):
        w = _weight(src, c["rows"], c["cols"], c["fmt"], exact=True)
        x = src.normal(c.get("batch", 1), c["cols"])
        out = (x.double() if kind == "logits" else _quantized(x)) @ w.T
        return out[0] if kind == "matvec" or kind == "logits" and c["batch"] == 1 else out
    kvd, qd = c["kv_heads"] * c["head_dim"], c["heads"] * c["head_dim"]
    if kind == "kvattn":
        k, v = src.normal(c["context"], kvd), src.normal(c["context"], kvd)
        q = src.normal(qd).double()[None]
        k, v = _cached(k, v, c["cache"], c["kv_heads"], c["head_dim"])
        return _attend(q, k, v, c["heads"], c["kv_heads"], c["head_dim"])[0]
    q, k, v = (src.normal(c["tokens"], n).double() for n in (qd, kvd, kvd))
    return _attend(q, k, v, c["heads"], c["kv_heads"], c["head_dim"])
