"""The work a user of this library has it do, as cases that can be timed and
checked: single q4 layers (the gather, linears from one row to a prompt, the
decode MLP), the two attention entry points, the reference's op-by-op
attention over strided tensors, and two whole calls of the decoder (one
captured decode step, one prompt).

A case is a dict of plain values. `prepare` builds what a user's program holds
before the call (weights, caches, tables, outputs it reuses, a captured step),
`run` makes one pass through the public entry points on the device's stream,
and `exact` restates the same result in plain float64 torch.

Shapes are those of the two decoders the library is configured for (hidden
3072 and 4096, 8 KV heads of 128), of smaller layers (hidden 2048, head size
64), and generic odd ones. Weights follow the library's q4 distribution:
uniform nibbles, scales U(0.004, 0.02), biases -8 s + N(0, 1e-3).
"""
import ctypes
import math

import torch

from foundry_amd import _lib
from foundry_amd.device import HipDevice, Layout
from foundry_amd.llama import LlamaConfig, Q4Llama, rope_tables
from foundry_amd.primitive import DType
from foundry_amd.tensor import Tensor

GROUP = 64

# hidden, query heads, KV heads, head size, FFN
SHAPES = {
    "h2048": (2048, 32, 8, 64, 8192),
    "h3072": (3072, 24, 8, 128, 8192),
    "h4096": (4096, 32, 8, 128, 14336),
}
VOCAB = 128256

_TORCH = {DType.F32: torch.float32, DType.BF16: torch.bfloat16, DType.U32: torch.int32}


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # a prompt batch's embedding rows: pure gather, write-dominated
        {"name": "embed_4096", "kind": "embed", "ids": 4096, "vocab": VOCAB, "k": 3072},
        # one token's gate/up projection: among the smallest calls, launch latency counts
        {"name": "linear_1", "kind": "linear", "rows": 1, "n": 16384, "k": 3072},
        # 32 concurrent sequences' gate/up projection: decode above the GEMV's 8 rows
        {"name": "linear_32", "kind": "linear", "rows": 32, "n": 28672, "k": 4096},
        # a 512-token prompt's q/k/v projection
        {"name": "linear_512", "kind": "linear", "rows": 512, "n": 5120, "k": 3072},
        # a 2048-token prompt's gate projection
        {"name": "linear_2048", "kind": "linear", "rows": 2048, "n": 8192, "k": 3072},
        # the MLP of 8 sequences' decode step: norm, gate/up, SiLU, down
        {"name": "mlp_8", "kind": "mlp", "rows": 8, "shape": "h4096"},
        # one sequence's decode attention at a long context
        {"name": "attn_decode_1", "kind": "attn_decode", "batch": 1, "shape": "h3072", "max_len": 4096, "pos": 4001},
        # 8 sequences' decode attention at a long context: the key/value stream
        {"name": "attn_decode_8", "kind": "attn_decode", "batch": 8, "shape": "h4096", "max_len": 4160, "pos": 4110},
        # a 2048-token prompt's attention after 1024 earlier tokens
        {"name": "attn_prompt_2048", "kind": "attn_prompt", "tokens": 2048, "past": 1024, "shape": "h4096"},
        # attention as the reference's unchanged model code runs it, op by op over strided views
        {"name": "attn_ops_512", "kind": "attn_ops", "tokens": 512, "past": 0, "shape": "h3072"},
        # a whole decode step (4 layers and the LM head), captured once and replayed per token
        {"name": "decode_step_1", "kind": "decode_step", "batch": 1, "layers": 4, "shape": "h3072", "max_len": 768,
         "pos": 640},
        # a whole 512-token prompt call (2 layers and the LM head)
        {"name": "prompt_512", "kind": "prompt", "tokens": 512, "layers": 2, "shape": "h3072"},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["embed", "linear", "linear", "linear", "mlp", "attn_decode", "attn_decode", "attn_prompt",
                       "attn_ops", "decode_step", "prompt"])
    name = rng.choice(sorted(SHAPES))
    hidden, heads, kv, hd, ffn = SHAPES[name]
    if kind == "embed":
        return {"kind": kind, "ids": _log(rng, 4096, 16384), "vocab": rng.randrange(30000, VOCAB + 1), "k": hidden}
    if kind == "linear":
        # a projection of a layer, or a generic size (n any, k a multiple of the group)
        n, k = rng.choice([((heads + 2 * kv) * hd, hidden), (hidden, heads * hd), (2 * ffn, hidden), (hidden, ffn),
                           (_log(rng, 1000, 16384), GROUP * _log(rng, 12, 160))])
        # (one row of a small projection takes less than 5 us)
        rows = _log(rng, 1 if n * k >= 40_000_000 else 2, 2048)
        most = 2048 * 8192 * 3072
        return {"kind": kind, "rows": max(1, min(rows, most // (n * k))), "n": n, "k": k}
    if kind == "mlp":
        return {"kind": kind, "rows": rng.randrange(1, 9), "shape": name}
    if kind == "attn_decode":
        max_len = _log(rng, 192, 4160)
        return {"kind": kind, "batch": rng.randrange(1, 9), "shape": name, "max_len": max_len,
                "pos": rng.randrange(max_len // 2, max_len)}
    if kind == "attn_prompt":
        return {"kind": kind, "tokens": _log(rng, 16, 2048), "past": rng.choice([0, _log(rng, 16, 1024)]),
                "shape": name}
    if kind == "attn_ops":
        return {"kind": kind, "tokens": _log(rng, 32, 512), "past": rng.choice([0, rng.randrange(1, 256)]),
                "shape": rng.choice(["h2048", "h3072"])}
    if kind == "decode_step":
        max_len = _log(rng, 256, 2048)
        return {"kind": kind, "batch": rng.randrange(1, 9), "layers": rng.randrange(1, 4), "shape": name,
                "max_len": max_len, "pos": rng.randrange(max_len // 2, max_len)}
    return {"kind": kind, "tokens": _log(rng, 9, 512), "layers": 1, "shape": name}


# ----------------------------------------------------------- device buffers

_device = None


def device():
    """One device object per process, as a user's program holds it."""
    global _device
    if _device is None:
        _device = HipDevice(0)
    return _device


class _Span:
    """A storage's memory as torch sees it; keeps the storage alive."""

    def __init__(self, storage, nbytes):
        self.storage = storage
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (storage.ptr, False),
                                         "version": 2}


def tensor_of(storage, dtype, shape):
    """The storage's first elements as a torch tensor on the same memory."""
    n = math.prod(shape) * torch.empty((), dtype=dtype).element_size()
    return torch.as_tensor(_Span(storage, n), device="cuda").view(dtype).view(shape)


def store(t):
    """A storage of the device holding t's values."""
    t = t.contiguous()
    st = device().empty(t.numel() * t.element_size())
    tensor_of(st, t.dtype, tuple(t.shape)).copy_(t)
    return st


def ptr(storage):
    return ctypes.c_void_p(storage.ptr)


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda").to(torch.bfloat16)


class Weight:
    """A q4 triplet: torch tensors, and the storages the library reads."""

    def __init__(self, g, n, k):
        self.n, self.k = n, k
        self.wq = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), generator=g, device="cuda", dtype=torch.int32)
        s = 0.004 + 0.016 * torch.rand((n, k // GROUP), generator=g, device="cuda")
        self.s = s.to(torch.bfloat16)
        z = torch.randn((n, k // GROUP), generator=g, device="cuda")
        self.b = (-8.0 * self.s.float() + 1e-3 * z).to(torch.bfloat16)
        st = [store(t) for t in (self.wq, self.s, self.b)]
        self.wq, self.s, self.b = [tensor_of(x, t.dtype, tuple(t.shape)) for x, t in zip(st, (self.wq, self.s, self.b))]
        self.ptrs = [ptr(x) for x in st]

    def exact(self):
        return dequant64(self.wq, self.s, self.b)


def dequant64(wq, s, b):
    """s * q + b in float64, [n, k]."""
    n = wq.shape[0]
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((wq.unsqueeze(-1) >> shifts) & 15).view(n, -1, GROUP).double()
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).view(n, -1)


def keys_of(k_cache, max_len, hd):
    """A K cache's memory [..., max_len * hd] (groups of 16 keys, laid out
    [hd / 32][keys][32]) as keys [..., max_len, hd]."""
    j = torch.arange(max_len, device="cuda").unsqueeze(1)
    d = torch.arange(hd, device="cuda").unsqueeze(0)
    n = torch.clamp(max_len - 16 * (j // 16), max=16)
    at = (j // 16) * 16 * hd + (d // 32) * n * 32 + (j % 16) * 32 + d % 32
    return k_cache.flatten(-2)[..., at.flatten()].view(*k_cache.shape[:-2], max_len, hd)


class State:
    """What prepare hands to run: `call` makes the pass, `out` is what it
    returns (buffers the pass writes), `inputs` what exact restates it from."""

    def __init__(self, call, out, inputs):
        self.call, self.out, self.inputs = call, out, inputs


# ------------------------------------------------------------------ prepare

def prepare(case, seed):
    return _PREPARE[case["kind"]](case, generator(seed), seed)


def run(state):
    got = state.call()
    return state.out if got is None else got


def _prepare_embed(c, g, seed):
    w = Weight(g, c["vocab"], c["k"])
    ids = torch.randint(0, c["vocab"], (c["ids"],), generator=g, device="cuda", dtype=torch.int32)
    ids_st, out = store(ids), device().empty(c["ids"] * c["k"] * 2)
    args = (device().handle, *w.ptrs, w.n, w.k, GROUP, ptr(ids_st), c["ids"], ptr(out))
    return State(lambda: _lib.call("fh_q4_embed", *args), tensor_of(out, torch.bfloat16, (c["ids"], c["k"])),
                 {"w": w, "ids": ids, "keep": ids_st})


def _prepare_linear(c, g, seed):
    m, n, k = c["rows"], c["n"], c["k"]
    w, x = Weight(g, n, k), normal(g, m, k)
    x_st, y = store(x), device().empty(m * n * 2)
    args = (device().handle, ptr(x_st), m, k, k, *w.ptrs, n, GROUP, ptr(y), _lib.BF16)
    return State(lambda: _lib.call("fh_q4_matmul", *args), tensor_of(y, torch.bfloat16, (m, n)),
                 {"w": w, "x": x, "keep": x_st})


def _prepare_mlp(c, g, seed):
    m = c["rows"]
    hidden, _, _, _, f = SHAPES[c["shape"]]
    up, down = Weight(g, 2 * f, hidden), Weight(g, hidden, f)
    x, h = normal(g, m, hidden), normal(g, m, hidden)
    norm = (1 + 0.1 * torch.randn(hidden, generator=g, device="cuda")).to(torch.bfloat16)
    st = [store(t) for t in (x, h, norm)]
    dev = device()
    h_out, act, y = dev.empty(m * hidden * 2), dev.empty(m * f * 2), dev.empty(m * hidden * 2)
    first = (dev.handle, ptr(st[0]), ptr(st[1]), ptr(h_out), ptr(st[2]), ctypes.c_float(1e-5), m, hidden, *up.ptrs,
             2 * f, GROUP, ptr(act))
    second = (dev.handle, ptr(act), m, f, f, *down.ptrs, hidden, GROUP, ptr(y), _lib.BF16)

    def call():
        _lib.call("fh_q4_gate_up_silu", *first)
        _lib.call("fh_q4_matmul", *second)

    bf = torch.bfloat16
    return State(call, {"h": tensor_of(h_out, bf, (m, hidden)), "act": tensor_of(act, bf, (m, f)),
                        "y": tensor_of(y, bf, (m, hidden))},
                 {"up": up, "down": down, "x": x, "h": h, "norm": norm, "keep": st})


def _rope(heads, kv, hd, length):
    cfg = LlamaConfig(n_layers=1, hidden=heads * hd, n_heads=heads, n_kv_heads=kv, head_dim=hd, ffn=64, vocab=16)
    return [torch.from_numpy(t.view("int16")).cuda().view(torch.bfloat16) for t in rope_tables(cfg, length)]


def _prepare_attn_decode(c, g, seed):
    _, heads, kv, hd, _ = SHAPES[c["shape"]]
    b, max_len, dev = c["batch"], c["max_len"], device()
    qkv = normal(g, b, (heads + 2 * kv) * hd)
    k, v = normal(g, b, kv, max_len, hd), normal(g, b, kv, max_len, hd)
    # sequences of one batch are at different depths
    pos = torch.tensor([max(0, c["pos"] - 17 * i) for i in range(b)], device="cuda", dtype=torch.int32)
    cos, sin = _rope(heads, kv, hd, max_len)
    st = [store(t) for t in (qkv, cos, sin, pos, k, v)]
    nbytes = _lib.decode_attention_workspace_bytes(b, heads, kv, hd, max_len)
    ws, out = dev.empty(nbytes), dev.empty(b * heads * hd * 2)
    args = (dev.handle, ptr(st[0]), b, heads, kv, hd, ptr(st[1]), ptr(st[2]), max_len, ptr(st[3]), ptr(st[4]),
            ptr(st[5]), max_len, ctypes.c_float(hd ** -0.5), ptr(ws), nbytes, ptr(out))
    bf = torch.bfloat16
    return State(lambda: _lib.call("fh_decode_attention", *args),
                 {"out": tensor_of(out, bf, (b, heads, hd)), "k": tensor_of(st[4], bf, (b, kv, max_len, hd)),
                  "v": tensor_of(st[5], bf, (b, kv, max_len, hd))},
                 {"qkv": qkv, "k": k, "v": v, "cos": cos, "sin": sin, "pos": pos, "keep": [st, ws]})


def _prepare_attn_prompt(c, g, seed):
    _, heads, kv, hd, _ = SHAPES[c["shape"]]
    t, max_len, dev = c["tokens"], c["past"] + c["tokens"], device()
    q, k, v = normal(g, t, heads, hd), normal(g, kv, max_len, hd), normal(g, kv, max_len, hd)
    pos = torch.arange(c["past"], max_len, device="cuda", dtype=torch.int32)
    st = [store(x) for x in (q, k, v, pos)]
    nbytes = _lib.attention_workspace_bytes(t, heads, kv, hd, max_len)
    ws, out = dev.empty(nbytes), dev.empty(t * heads * hd * 2)
    args = (dev.handle, *[ptr(s) for s in st], t, heads, kv, hd, max_len, ctypes.c_float(hd ** -0.5), ptr(ws), nbytes,
            ptr(out))
    return State(lambda: _lib.call("fh_attention", *args), tensor_of(out, torch.bfloat16, (t, heads, hd)),
                 {"q": q, "k": k, "v": v, "past": c["past"], "keep": [st, ws]})


def _tensor(t, dtype):
    return Tensor(store(t), Layout.contiguous(tuple(t.shape)), dtype)


def _prepare_attn_ops(c, g, seed):
    _, heads, kv, hd, _ = SHAPES[c["shape"]]
    t, ctx, dev, group = c["tokens"], c["past"] + c["tokens"], device(), heads // kv
    q, k, v = normal(g, t, heads, hd), normal(g, kv, ctx, hd), normal(g, kv, ctx, hd)
    mask = torch.full((t, ctx), -math.inf, device="cuda").triu(c["past"] + 1)
    qt, kt, vt = _tensor(q, DType.BF16), _tensor(k, DType.BF16), _tensor(v, DType.BF16)
    mt, scale = _tensor(mask, DType.F32), Tensor.scalar_f32(dev, hd ** -0.5)

    def call():
        # q [t, heads, hd] read in place as [kv, group, t, hd]; keys and
        # values broadcast over the heads that share them
        qv = qt.reshape((t, kv, group, hd)).permute((1, 2, 0, 3))
        kv_t = kt.reshape((kv, 1, ctx, hd)).expand((kv, group, ctx, hd)).permute((0, 1, 3, 2))
        vv = vt.reshape((kv, 1, ctx, hd)).expand((kv, group, ctx, hd))
        s = qv.matmul(dev, kv_t).to_dtype(dev, DType.F32).mul(dev, scale).add(dev, mt)
        e = s.sub(dev, s.amax_keepdim(dev, 3)).exp(dev)
        p = e.div(dev, e.sum_keepdim(dev, 3)).to_dtype(dev, DType.BF16)
        o = p.matmul(dev, vv).permute((2, 0, 1, 3)).contiguous(dev)
        return tensor_of(o.storage, torch.bfloat16, (t, heads, hd))

    return State(call, None, {"q": q, "k": k, "v": v, "past": c["past"]})


def _config(c):
    hidden, heads, kv, hd, ffn = SHAPES[c["shape"]]
    return LlamaConfig(c["layers"], hidden, heads, kv, hd, ffn, VOCAB)


def _model(c, max_len, max_tokens, batch, g):
    """A decoder whose weights the library draws once per shape, refilled
    here from the case's seed: new words per layer, and (through the
    library's own calls) the copies it keeps of them."""
    m = Q4Llama(device(), _config(c), 0, max_len, max_tokens, batch)
    device().synchronize()
    for w in [m.embed] + [layer[key] for layer in m.layers for key in ("qkv", "o", "gate_up", "down")]:
        words = tensor_of(w.wq, torch.int32, (w.n, w.k // 8))
        words.random_(-2 ** 31, 2 ** 31, generator=g)
    torch.cuda.synchronize()
    for layer in m.layers + [{"embed": m.embed}]:
        for key in ("qkv", "o", "gate_up", "down", "embed"):
            w = layer.get(key)
            if w is not None and w.wt is not None:
                _lib.call("fh_q4_tile", device().handle, ptr(w.wq), w.n, w.k, GROUP, int(key == "gate_up"), ptr(w.wt))
    return m


def _fill_caches(m, g):
    cfg, out = m.cfg, []
    for layer in m.layers:
        for key in ("k_cache", "v_cache"):
            t = tensor_of(layer[key], torch.bfloat16, (m.batch, cfg.n_kv_heads, m.max_len, cfg.head_dim))
            t.copy_(normal(g, *t.shape))
            out.append(t)
    return out


def _logits(m):
    return tensor_of(m.buf["logits"], torch.bfloat16, (m.batch, m.cfg.vocab))


# The decoder's outputs are its logits and caches. The greedy id beside them
# is the first largest logit: all or nothing under a tie, so not compared.

def _prepare_decode_step(c, g, seed):
    dev, b = device(), c["batch"]
    m = _model(c, c["max_len"], 1, b, g)
    caches = _fill_caches(m, g)
    ids = torch.randint(0, VOCAB, (b,), generator=g, device="cuda", dtype=torch.int32)
    pos = torch.tensor([max(0, c["pos"] - 17 * i) for i in range(b)], device="cuda", dtype=torch.int32)
    st = [store(ids), store(pos)]
    before = [t.clone() for t in caches]
    torch.cuda.synchronize()
    dev.capture_begin()
    _lib.call("fh_llama_forward", dev.handle, ctypes.addressof(m._model), 1, ptr(st[0]), ptr(st[1]), ptr(m.buf["next"]))
    graph = dev.capture_end()
    return State(graph.launch, {"logits": _logits(m), "caches": caches},
                 {"m": m, "ids": ids.view(b, 1), "pos": pos.view(b, 1), "caches": before, "keep": [st, graph]})


def _prepare_prompt(c, g, seed):
    t = c["tokens"]
    m = _model(c, t, t, 1, g)
    ids = torch.randint(0, VOCAB, (1, t), generator=g, device="cuda", dtype=torch.int32)
    prompt = ids.cpu().numpy().astype("uint32")
    caches = [tensor_of(layer[key], torch.bfloat16, (1, m.cfg.n_kv_heads, t, m.cfg.head_dim))
              for layer in m.layers for key in ("k_cache", "v_cache")]
    return State(lambda: m.prefill(prompt), {"logits": _logits(m), "caches": caches},
                 {"m": m, "ids": ids, "pos": torch.arange(t, device="cuda").view(1, t), "caches": caches})


_PREPARE = {"embed": _prepare_embed, "linear": _prepare_linear, "mlp": _prepare_mlp,
            "attn_decode": _prepare_attn_decode, "attn_prompt": _prepare_attn_prompt, "attn_ops": _prepare_attn_ops,
            "decode_step": _prepare_decode_step, "prompt": _prepare_prompt}


# --------------------------------------------------------------------- work

def _q4_bytes(n, k):
    return n * k // 2 + 4 * n * (k // GROUP)


def _linear_work(m, n, k):
    return _q4_bytes(n, k) + 2 * m * (n + k), 2 * m * n * k


def work(case):
    c = case
    hidden, heads, kv, hd, f = SHAPES[c.get("shape", "h3072")]
    if c["kind"] == "embed":
        per_id = c["k"] // 2 + 4 * (c["k"] // GROUP) + 4 + 2 * c["k"]
        return {"bytes": c["ids"] * per_id, "flops": 2 * c["ids"] * c["k"]}
    if c["kind"] == "linear":
        nbytes, flops = _linear_work(c["rows"], c["n"], c["k"])
    elif c["kind"] == "mlp":
        m = c["rows"]
        nbytes = _q4_bytes(2 * f, hidden) + _q4_bytes(hidden, f) + 2 * m * (4 * hidden + f)
        flops = 6 * m * f * hidden
    elif c["kind"] == "attn_decode":
        keys = sum(max(0, c["pos"] - 17 * i) + 1 for i in range(c["batch"]))
        nbytes = 4 * keys * kv * hd + 4 * c["batch"] * (heads + kv) * hd
        flops = 4 * keys * heads * hd
    elif c["kind"] in ("attn_prompt", "attn_ops"):
        t, past = c["tokens"], c["past"]
        nbytes = 4 * t * heads * hd + 4 * (past + t) * kv * hd
        flops = 4 * heads * hd * (t * past + t * (t + 1) // 2)
    else:
        seqs, t = c.get("batch", 1), c.get("tokens", 1)
        keys = (sum(max(0, c["pos"] - 17 * i) + 1 for i in range(seqs)) if c["kind"] == "decode_step"
                else t * (t + 1) // 2)
        seen = keys if c["kind"] == "decode_step" else t
        layer = [((heads + 2 * kv) * hd, hidden), (hidden, heads * hd), (2 * f, hidden), (hidden, f)]
        nbytes = _q4_bytes(VOCAB, hidden) + seqs * 2 * VOCAB
        nbytes += c["layers"] * (sum(_q4_bytes(n, k) for n, k in layer) + 4 * seen * kv * hd)
        flops = 2 * seqs * VOCAB * hidden
        flops += c["layers"] * (sum(2 * seqs * t * n * k for n, k in layer) + 4 * keys * heads * hd)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Relative errors of bf16 results: one rounding of the output for the
    linears, one more per bf16 intermediate (the MLP's activations, the
    attention's scores and probabilities), and each layer's for the decoder.
    Each is about four times the error measured against `exact`."""
    return {"embed": "exact", "linear": {"rel": 8e-3}, "mlp": {"rel": 1.5e-2}, "attn_decode": {"rel": 1.5e-2},
            "attn_prompt": {"rel": 1.5e-2}, "attn_ops": {"rel": 1.5e-2}, "decode_step": {"rel": 1.5e-2},
            "prompt": {"rel": 1.5e-2}}[case["kind"]]


# -------------------------------------------------------------------- exact

def exact(case, seed):
    s = prepare(case, seed)
    torch.cuda.synchronize()
    device().synchronize()
    return _EXACT[case["kind"]](s.inputs)


def _exact_embed(i):
    return dequant64(*[t[i["ids"].long()] for t in (i["w"].wq, i["w"].s, i["w"].b)])


def _exact_linear(i):
    return i["x"].double() @ i["w"].exact().T


def _norm64(h, w):
    return h / torch.sqrt(h.square().mean(-1, keepdim=True) + 1e-5) * w.double()


def _mlp64(x, up, down):
    gate, lin = (x @ up.T).chunk(2, -1)
    act = gate / (1 + torch.exp(-gate)) * lin
    return act, act @ down.T


def _exact_mlp(i):
    h = i["x"].double() + i["h"].double()
    act, y = _mlp64(_norm64(h, i["norm"]), i["up"].exact(), i["down"].exact())
    return {"h": h, "act": act, "y": y}


def _rotate64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos + torch.cat([-b, a], -1) * sin


def _attend64(q, k, v, pos):
    """q [t, heads, hd] at positions pos over k, v [kv, keys, hd]."""
    t, heads, hd = q.shape
    group = heads // k.shape[0]
    out = torch.empty(t, heads, hd, device="cuda", dtype=torch.float64)
    ahead = torch.arange(k.shape[1], device="cuda").unsqueeze(0) > pos.view(t, 1)
    for h in range(heads):
        s = (q[:, h] @ k[h // group].T * hd ** -0.5).masked_fill(ahead, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[h // group]
    return out


def _exact_attn_decode(i):
    b, kv, max_len, hd = i["k"].shape
    heads = i["qkv"].shape[1] // hd - 2 * kv
    keys, values = keys_of(i["k"], max_len, hd).double(), i["v"].double()
    out = []
    for n in range(b):
        p = int(i["pos"][n])
        x = i["qkv"][n].double().view(-1, hd)
        rot = _rotate64(x[:heads + kv], i["cos"][p].double(), i["sin"][p].double())
        keys[n, :, p], values[n, :, p] = rot[heads:], x[heads + kv:]
        out.append(_attend64(rot[None, :heads], keys[n], values[n], i["pos"][n:n + 1]))
    return {"out": torch.cat(out), "k": None, "v": None}


def _exact_attn_prompt(i):
    k = keys_of(i["k"], *i["k"].shape[1:]).double()
    pos = i["past"] + torch.arange(i["q"].shape[0], device="cuda")
    return _attend64(i["q"].double(), k, i["v"].double(), pos)


def _exact_attn_ops(i):
    pos = i["past"] + torch.arange(i["q"].shape[0], device="cuda")
    return _attend64(i["q"].double(), i["k"].double(), i["v"].double(), pos)


def _exact_decoder(i):
    m = i["m"]
    c = m.cfg
    heads, kv, hd = c.n_heads, c.n_kv_heads, c.head_dim
    bf = torch.bfloat16

    def weight(w, rows=slice(None)):
        g = w.k // GROUP
        return dequant64(tensor_of(w.wq, torch.int32, (w.n, w.k // 8))[rows], tensor_of(w.s, bf, (w.n, g))[rows],
                         tensor_of(w.b, bf, (w.n, g))[rows])

    seqs, t = i["ids"].shape
    pos = i["pos"].long()
    cos, sin = [tensor_of(s, bf, (m.max_len, hd)).double()[pos].unsqueeze(2) for s in (m.cos, m.sin)]
    h = weight(m.embed, i["ids"].long().flatten()).view(seqs, t, c.hidden)
    for n, layer in enumerate(m.layers):
        norm = [tensor_of(layer[key], bf, (c.hidden,)) for key in ("input_norm", "post_norm")]
        x = (_norm64(h, norm[0]) @ weight(layer["qkv"]).T).view(seqs, t, heads + 2 * kv, hd)
        rot = _rotate64(x[:, :, :heads + kv], cos, sin)
        attn = torch.empty(seqs, t, heads, hd, device="cuda", dtype=torch.float64)
        for q in range(seqs):
            k = keys_of(i["caches"][2 * n][q], m.max_len, hd).double()
            v = i["caches"][2 * n + 1][q].double()
            k[:, pos[q]] = rot[q, :, heads:].transpose(0, 1)
            v[:, pos[q]] = x[q, :, heads + kv:].transpose(0, 1)
            attn[q] = _attend64(rot[q, :, :heads], k, v, pos[q])
        h = h + attn.flatten(-2) @ weight(layer["o"]).T
        _, y = _mlp64(_norm64(h, norm[1]), weight(layer["gate_up"]), weight(layer["down"]))
        h = h + y
    last = _norm64(h[:, -1], tensor_of(m.final_norm, bf, (c.hidden,)))
    parts = [last @ weight(m.embed, slice(r, r + 16384)).T for r in range(0, c.vocab, 16384)]
    return {"logits": torch.cat(parts, -1), "caches": [None] * len(i["caches"])}


_EXACT = {"embed": _exact_embed, "linear": _exact_linear, "mlp": _exact_mlp, "attn_decode": _exact_attn_decode,
          "attn_prompt": _exact_attn_prompt, "attn_ops": _exact_attn_ops, "decode_step": _exact_decoder,
          "prompt": _exact_decoder}
