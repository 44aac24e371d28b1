"""Performance cases of the quantized-weight path on one GPU.

Each case is work that a program using the package has it do through its
public entry points: the linear layers of one decoder layer over T token rows
(`Gfx950Backend.rmsnorm`, `qmatmul_qkv`, `qmatmul`, `add_rmsnorm`,
`ffn_gate_up`, `add`), attention over a KV cache (`attn`), the output head
(`qmatmul`, `greedy`), and whole models (`Session.prefill`,
`Decoder.forward`). Geometries are those of `mdma_amd.llama_synth`
(TinyStories-15M, Llama-3-8B) and generic ones between them.

Weights are GGUF blocks whose dequantized values are about N(0, 0.02), as in a
trained model; activations are a residual stream with a few channels much
larger than the rest.
"""
import math
import os
import tempfile

import numpy as np
import torch

from mdma_amd import gguf, llama_synth
from mdma_amd.backend import (ACT_F32, ACT_F32_CPU, ACT_I8, GGML_F32, GGML_Q4_K, GGML_Q6_K, GGML_Q8_0, AttnSpec,
                              Gfx950Backend, KvView)
from mdma_amd.model import Model

MODES = {"f32": ACT_F32, "int8": ACT_I8, "cpu": ACT_F32_CPU}
EPS = 1e-5
# Weight types of a layer's matrices (qkv, o, gate/up, down).
MIXES = {"Q4_K": (GGML_Q4_K,) * 4, "Q4_K_M": (GGML_Q6_K, GGML_Q6_K, GGML_Q4_K, GGML_Q6_K), "Q8_0": (GGML_Q8_0,) * 4}
BITS = {GGML_Q4_K: 4.5, GGML_Q6_K: 6.5625, GGML_Q8_0: 8.5, GGML_F32: 32.0}

L8B = dict(embd=4096, heads=32, kv_heads=8, ff=14336)
TINY = dict(embd=288, heads=6, kv_heads=6, ff=768)
# Widths between the two: whole 256-column blocks, not all powers of two.
MID = (dict(embd=2048, heads=32, kv_heads=8, ff=5632), dict(embd=2560, heads=20, kv_heads=20, ff=6912),
       dict(embd=3072, heads=24, kv_heads=8, ff=8192))


def _linears(name, mix, mode, tokens, geom):
    c = dict(kind="linears", mix=mix, mode=mode, tokens=tokens, **geom)
    return dict(c, name=name) if name else c


def _attn(name, mode, queries, keys, heads, kv_heads, head_dim):
    c = dict(kind="attn", mode=mode, queries=queries, keys=keys, heads=heads, kv_heads=kv_heads, head_dim=head_dim)
    return dict(c, name=name) if name else c


def _model(name, geom, mode, step, tokens):
    c = dict(kind="model", geom=geom, mode=mode, step=step, tokens=tokens)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The smallest whole call: one greedy step of the TinyStories-15M geometry (all Q8_0) in the default
        # mode, replayed by the graph decoder, logits to the host. Launches and latency.
        _model("tiny_decode_f32", "tiny", "f32", "decode", 100),
        # Token by token generation with Llama-3-8B (Q4_K_M): one layer's projections for one token, captured
        # into a graph as a decoder replays them; int8 activations.
        _linears("decode1_int8", "Q4_K_M", "int8", 1, L8B),
        # The same step in the default (f32) mode.
        _linears("decode1_f32", "Q4_K_M", "f32", 1, L8B),
        # Eight sequences decoded together.
        _linears("decode8_int8", "Q4_K_M", "int8", 8, L8B),
        # The end of a decode step: final norm, the 128256-row head, the greedy token on the host.
        dict(name="head_int8", kind="head", mode="int8", dtype="Q6_K", vocab=128256, embd=4096, tokens=1),
        # A short prompt (a chat turn), a ragged number of tokens.
        _linears("prompt43_int8", "Q4_K_M", "int8", 43, L8B),
        # A 512-token prompt through the model driver: embedding, two layers of the Llama-3-8B geometry with
        # attention, the head on the last row.
        _model("prefill512_int8", "l8b2", "int8", "prefill", 512),
        # A long prompt on an all-Q8_0 model.
        _linears("prompt2048_q8_int8", "Q8_0", "int8", 2048, L8B),
        # A prompt in the default mode, f32 activations.
        _linears("prompt300_f32", "Q4_K_M", "f32", 300, L8B),
        # Attention of a long prompt's second half (causal, over a prefix).
        _attn("attn_prompt1500", "f32", 1500, 2500, 32, 8, 128),
        # Attention of one decoded token late in a 4096-token context.
        _attn("attn_decode3900", "f32", 1, 3900, 32, 8, 128),
        # One decode step's projections in the mode that reproduces the CPU backend bit for bit.
        _linears("decode1_cpu", "Q4_K_M", "cpu", 1, L8B),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linears"] * 6 + ["attn"] * 2 + ["head", "model"])
    if kind == "linears":
        mode = rng.choice(["int8", "int8", "int8", "f32", "f32", "cpu"])
        geom = rng.choice([L8B, L8B, L8B, *MID, TINY])
        mix = "Q8_0" if geom is TINY else rng.choice(["Q4_K_M", "Q4_K_M", "Q4_K", "Q8_0"])
        hi = {"int8": 1800, "f32": 300, "cpu": 4}[mode]
        return _linears(None, mix, mode, _log_int(rng, 1, hi), geom)
    if kind == "attn":
        heads, kv_heads, head_dim = rng.choice([(32, 8, 128), (32, 8, 128), (32, 32, 64), (20, 20, 128), (6, 6, 48)])
        queries = _log_int(rng, 1, 1500 if head_dim >= 64 else 100)
        keys = queries + rng.choice([0, _log_int(rng, 1, 2500 if queries > 64 else 4000 - queries)])
        return _attn(None, "f32", queries, keys, heads, kv_heads, head_dim)
    if kind == "head":
        return dict(kind="head", mode=rng.choice(["int8", "f32"]), dtype=rng.choice(["Q6_K", "Q8_0"]),
                    vocab=rng.choice([32000, 32001, 49152, 100352]), embd=rng.choice([2048, 2560, 4096]),
                    tokens=rng.choice([1, 1, 1, 4, 8]))
    step = rng.choice(["prefill", "decode"])
    return _model(None, "tiny", rng.choice(["f32", "int8"]), step, _log_int(rng, 4, 200))


# ---- seeded inputs, made on the GPU ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _randint(g, lo, hi, *shape):
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=torch.int32)


def _f16_bytes(t):
    return t.to(torch.float16).view(torch.uint8).reshape(t.shape[0], -1)


def _blocks(g, dtype, rows, cols, sigma=0.02):
    """GGUF blocks of a [rows, cols] weight whose values are about N(0, sigma): uint8 [blocks, block bytes]."""
    if dtype == GGML_Q8_0:
        n = rows * cols // 32
        q = (_randn(g, n, 32) * 45).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        d = sigma / 45 * (0.7 + 0.6 * torch.rand(n, generator=g, device="cuda"))
        return torch.cat([_f16_bytes(d[:, None]), q], 1)
    n = rows * cols // 256
    spread = (0.7 + 0.6 * torch.rand(n, generator=g, device="cuda"))[:, None]
    if dtype == GGML_Q4_K:
        sc = _randint(g, 24, 63, n, 8)
        m = (sc + _randint(g, -6, 6, n, 8)).clamp(0, 63)
        q = (_randn(g, n, 256) * 3.2 + 7.5).round().clamp(0, 15).to(torch.uint8)
        d = sigma / (3.2 * 43) * spread
        scb = torch.empty(n, 12, dtype=torch.int32, device="cuda")
        scb[:, 0:4] = sc[:, 0:4] | ((sc[:, 4:8] >> 4) << 6)
        scb[:, 4:8] = m[:, 0:4] | ((m[:, 4:8] >> 4) << 6)
        scb[:, 8:12] = (sc[:, 4:8] & 15) | ((m[:, 4:8] & 15) << 4)
        qs = q.view(n, 4, 2, 32)
        return torch.cat([_f16_bytes(d), _f16_bytes(7.5 * d), scb.to(torch.uint8),
                          (qs[:, :, 0] | (qs[:, :, 1] << 4)).reshape(n, 128)], 1)
    q = (_randn(g, n, 256) * 11).round().clamp(-32, 31).to(torch.int32) + 32
    sc = (_randint(g, 40, 127, n, 16) * (1 - 2 * _randint(g, 0, 1, n, 16))).to(torch.int8).view(torch.uint8)
    d = sigma / (11 * 85) * spread
    v = q.view(n, 2, 4, 32)  # half, quarter, column
    ql = torch.stack([(v[:, :, 0] & 15) | ((v[:, :, 2] & 15) << 4), (v[:, :, 1] & 15) | ((v[:, :, 3] & 15) << 4)], 2)
    qh = sum((v[:, :, r] >> 4) << (2 * r) for r in range(4))
    return torch.cat([ql.reshape(n, 128).to(torch.uint8), qh.reshape(n, 64).to(torch.uint8), sc, _f16_bytes(d)], 1)


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(blk, dtype, rows, cols):
    """The values of GGUF blocks in 64 bits: [rows, cols]."""
    n = blk.shape[0]
    if dtype == GGML_Q8_0:
        return (_half(blk[:, 0:2]) * blk[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if dtype == GGML_Q4_K:
        s = blk[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = blk[:, 16:].view(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).double()
        return ((_half(blk[:, 0:2]) * sc)[:, :, None] * q - (_half(blk[:, 2:4]) * m)[:, :, None]).reshape(rows, cols)
    ql, qh = blk[:, 0:128].view(n, 2, 2, 32), blk[:, 128:192].view(n, 2, 32)
    quarters = [(ql[:, :, r & 1] >> (4 * (r >> 1)) & 15).to(torch.int32) | ((qh >> (2 * r) & 3).to(torch.int32) << 4)
                for r in range(4)]
    q = torch.stack(quarters, 2).reshape(n, 16, 16).double() - 32
    sc = blk[:, 192:208].contiguous().view(torch.int8).double()
    return ((_half(blk[:, 208:210]) * sc)[:, :, None] * q).reshape(rows, cols)


def _stream(g, tokens, embd):
    """A residual stream: N(0, 1) with one channel in about 200 fifteen times larger."""
    big = 1 + 14 * (torch.rand(embd, generator=g, device="cuda") < 0.005)
    return _randn(g, tokens, embd) * big


def _norm_weight(g, embd):
    return 1 + 0.1 * _randn(g, embd)


# ---- the package's side ----

_backends = {}


def _backend(mode):
    """One context per activation mode, as a program keeps one for its device."""
    if mode not in _backends:
        be = Gfx950Backend(0)
        be.set_act_mode(MODES[mode])
        _backends[mode] = be
    return _backends[mode]


def _upload(be, t):
    return be.f32_buf(t.detach().cpu().numpy())


def _weight(be, blk, dtype, rows, cols):
    return be.upload_weight(blk.cpu().numpy().reshape(-1), dtype, (rows, cols))


class Outputs(dict):
    """Device buffers by name, each read to the host as float32 when looked at (the calls that fill them are
    queued on the backend's stream, and a program reads a result when it needs it)."""

    def __init__(self, be, bufs):
        super().__init__(bufs)
        self.be = be

    def __getitem__(self, name):
        buf, shape = dict.__getitem__(self, name)
        return self.be.download_f32(buf, math.prod(shape)).reshape(shape)


def _layer_shapes(c):
    E, F = c["embd"], c["ff"]
    hd = E // c["heads"]
    qd, kd = c["heads"] * hd, c["kv_heads"] * hd
    qkv, o, gu, down = MIXES[c["mix"]]
    return {"q": (qkv, qd, E), "k": (qkv, kd, E), "v": (qkv, kd, E), "o": (o, E, qd), "gate": (gu, F, E),
            "up": (gu, F, E), "down": (down, E, F)}


def _linears_inputs(c, seed):
    g = _gen(seed)
    T, E = c["tokens"], c["embd"]
    shapes = _layer_shapes(c)
    blks = {k: _blocks(g, dt, r, n) for k, (dt, r, n) in shapes.items()}
    acts = {"x": _stream(g, T, E), "att": 0.5 * _randn(g, T, shapes["o"][2]), "w1": _norm_weight(g, E),
            "w2": _norm_weight(g, E)}
    return shapes, blks, acts


def _linears_prepare(c, seed):
    be = _backend(c["mode"])
    shapes, blks, acts = _linears_inputs(c, seed)
    T = c["tokens"]
    s = {"be": be, "kind": "linears", "w": {k: _weight(be, blks.pop(k), *shapes[k]) for k in shapes},
         "a": {k: _upload(be, v) for k, v in acts.items()}, "graph": None}
    rows = {k: shapes[k][1] for k in ("q", "k", "v", "gate", "up")}
    rows.update(normed=c["embd"], proj=c["embd"], sum=c["embd"], act=c["ff"], ffn=c["embd"], out=c["embd"])
    s["b"] = {k: be.alloc(T * n * 4) for k, n in rows.items()}
    s["out"] = Outputs(be, {k: (s["b"][k], (T, rows[k])) for k in ("q", "k", "v", "proj", "ffn", "out")})
    if T <= 16:  # decode: the step is captured once and replayed, as a decoder does
        _linears_step(s)
        be.join_execution()
        s["graph"] = be.capture(lambda: _linears_step(s))
    return s


def _linears_step(s):
    be, w, a, b = s["be"], s["w"], s["a"], s["b"]
    be.rmsnorm(a["w1"], a["x"], b["normed"], EPS)
    be.qmatmul_qkv(w["q"], w["k"], w["v"], b["normed"], b["q"], b["k"], b["v"])
    be.qmatmul(w["o"], a["att"], b["proj"])
    be.add_rmsnorm(a["w2"], a["x"], b["proj"], b["sum"], b["normed"], EPS)
    be.ffn_gate_up(w["gate"], w["up"], b["normed"], b["gate"], b["up"], b["act"])
    be.qmatmul(w["down"], b["act"], b["ffn"])
    be.add(b["sum"], b["ffn"], b["out"])


def _attn_inputs(c, seed):
    g = _gen(seed)
    hd = c["head_dim"]
    q = _randn(g, c["queries"], c["heads"] * hd)
    k = (_randn(g, c["keys"], c["kv_heads"] * hd) * 0.8).to(torch.float16)
    v = _randn(g, c["keys"], c["kv_heads"] * hd).to(torch.float16)
    return q, k, v


def _attn_prepare(c, seed):
    be = _backend(c["mode"])
    q, k, v = _attn_inputs(c, seed)
    s = {"be": be, "kind": "attn", "q": _upload(be, q), "o": be.alloc(q.numel() * 4)}
    for n, t in (("k", k), ("v", v)):
        s[n] = be.alloc(t.numel() * 2)
        be.upload(s[n], 0, t.cpu().numpy())
    s["kv"] = KvView(s["k"], s["v"], c["keys"])
    s["spec"] = AttnSpec(c["head_dim"], c["heads"], c["kv_heads"])
    s["out"] = Outputs(be, {"o": (s["o"], tuple(q.shape))})
    return s


def _head_inputs(c, seed):
    g = _gen(seed)
    dt = {"Q6_K": GGML_Q6_K, "Q8_0": GGML_Q8_0}[c["dtype"]]
    return dt, _blocks(g, dt, c["vocab"], c["embd"]), _stream(g, c["tokens"], c["embd"]), _norm_weight(g, c["embd"])


def _head_prepare(c, seed):
    be = _backend(c["mode"])
    dt, blk, x, w = _head_inputs(c, seed)
    s = {"be": be, "kind": "head", "w": _weight(be, blk, dt, c["vocab"], c["embd"]), "x": _upload(be, x),
         "norm": _upload(be, w), "normed": be.alloc(x.numel() * 4), "logits": be.alloc(c["tokens"] * c["vocab"] * 4),
         "vocab": c["vocab"], "tokens": c["tokens"]}
    s["out"] = Outputs(be, {"logits": (s["logits"], (c["tokens"], c["vocab"]))})
    return s


def _model_geom(c):
    if c["geom"] == "tiny":
        return dict(llama_synth.TINYSTORIES), dict(llama_synth.Q8_ALL)
    # The Llama-3-8B geometry, two of its layers and a quarter of its vocabulary.
    return dict(llama_synth.LLAMA3_8B, n_layers=2, vocab=32000), dict(llama_synth.Q4_K_M)


def _model_tensors(geom, dtypes, g):
    """(name, dtype, shape, uint8 blocks or float32 values on the GPU) in load order."""
    def make(name, dtype, shape):
        if len(shape) == 1:
            return _norm_weight(g, shape[0])
        if dtype == GGML_F32:
            return _randn(g, *shape) * 0.02
        return _blocks(g, dtype, *shape)
    for name, dtype, shape, _ in llama_synth.tensors(geom, dtypes, 0):
        yield name, dtype, shape, make(name, dtype, shape)


class _ModelState:
    """A loaded model, its session and its decoder, released together."""

    def __init__(self, be, path, capacity, max_tokens, decode):
        self.model = Model(be, path)
        self.session = self.model.session(capacity, 1, max_tokens)
        self.decoder = self.session.decoder() if decode else None

    def __del__(self):
        for h in (self.decoder, self.session, self.model):
            if h is not None:
                h.close()


def _model_inputs(c, seed):
    geom, dtypes = _model_geom(c)
    g = _gen(seed)
    toks = _randint(g, 0, geom["vocab"] - 1, c["tokens"] + 1).cpu().numpy().astype(np.uint32)
    return geom, dtypes, toks, _model_tensors(geom, dtypes, g)


def _model_prepare(c, seed):
    be = _backend(c["mode"])
    geom, dtypes, toks, tensors = _model_inputs(c, seed)
    payload = [(n, dt, sh, t.cpu().numpy()) for n, dt, sh, t in tensors]
    fd, path = tempfile.mkstemp(suffix=".gguf")
    os.close(fd)
    try:
        gguf.write_stream(path, llama_synth.metadata(geom), [(n, dt, sh, lambda t=t: t) for n, dt, sh, t in payload])
        m = _ModelState(be, path, min(geom["n_ctx"], 4096), c["tokens"], c["step"] == "decode")
    finally:
        os.unlink(path)
    s = {"be": be, "kind": "model", "m": m, "toks": toks, "step": c["step"], "pos": c["tokens"]}
    if c["step"] == "decode":
        m.session.prefill(toks[:-1])
        m.decoder.forward(int(toks[-1]), c["tokens"])  # captures the step
    return s


def prepare(case, seed):
    return {"linears": _linears_prepare, "attn": _attn_prepare, "head": _head_prepare,
            "model": _model_prepare}[case["kind"]](case, seed)


def run(s):
    be = s["be"]
    if s["kind"] == "linears":
        if s["graph"] is not None:
            s["graph"].launch()
        else:
            _linears_step(s)
        return s["out"]
    if s["kind"] == "attn":
        be.attn(s["q"], s["kv"], s["spec"], s["o"])
        return s["out"]
    if s["kind"] == "head":
        be.rmsnorm(s["norm"], s["x"], s["normed"], EPS)
        be.qmatmul(s["w"], s["normed"], s["logits"])
        tokens = [be.greedy(s["logits"], t * s["vocab"], s["vocab"]) for t in range(s["tokens"])]
        return [s["out"], tokens]
    if s["step"] == "decode":
        return {"logits": s["m"].decoder.forward(int(s["toks"][-1]), s["pos"])}
    s["m"].session.reset()
    return {"logits": s["m"].session.prefill(s["toks"][:-1])}


# ---- what a pass cannot do without ----

def _layer_work(shapes, T, extra):
    w = sum(r * n * BITS[dt] / 8 for dt, r, n in shapes.values())
    flops = 2.0 * T * sum(r * n for _, r, n in shapes.values())
    return w + 4.0 * T * extra, flops


def _attn_flops(queries, keys, heads, hd):
    pairs = queries * (keys - queries) + queries * (queries + 1) / 2
    return 4.0 * pairs * heads * hd


def work(case):
    c = case
    if c["kind"] == "linears":
        sh = _layer_shapes(c)
        # x and att read; q, k, v, proj, ffn and out written.
        b, f = _layer_work(sh, c["tokens"], c["embd"] * 4 + sh["q"][1] * 2 + 2 * sh["k"][1])
        return {"bytes": b, "flops": f}
    if c["kind"] == "attn":
        qd, kd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        return {"bytes": 8.0 * c["queries"] * qd + 4.0 * c["keys"] * kd,
                "flops": _attn_flops(c["queries"], c["keys"], c["heads"], c["head_dim"])}
    if c["kind"] == "head":
        bits = BITS[{"Q6_K": GGML_Q6_K, "Q8_0": GGML_Q8_0}[c["dtype"]]]
        return {"bytes": c["vocab"] * c["embd"] * bits / 8 + 4.0 * c["tokens"] * (c["embd"] + c["vocab"]),
                "flops": 2.0 * c["tokens"] * c["vocab"] * c["embd"]}
    geom, dtypes = _model_geom(c)
    T, keys = (1, c["tokens"] + 1) if c["step"] == "decode" else (c["tokens"], c["tokens"])
    E, V, F, L = geom["n_embd"], geom["vocab"], geom["n_ff"], geom["n_layers"]
    hd = E // geom["n_heads"]
    kd = geom["n_kv_heads"] * hd
    mats = [("attn_q", E, E), ("attn_k", kd, E), ("attn_v", kd, E), ("attn_output", E, E), ("ffn_gate", F, E),
            ("ffn_up", F, E), ("ffn_down", E, F)]
    b = L * sum(r * n * BITS[dtypes[k]] / 8 for k, r, n in mats) + V * E * BITS[dtypes["output"]] / 8
    b += T * E * BITS[dtypes["token_embd"]] / 8 + 4.0 * V + L * 4.0 * keys * kd
    f = L * (2.0 * T * sum(r * n for _, r, n in mats) + _attn_flops(T, keys, geom["n_heads"], hd)) + 2.0 * V * E
    return {"bytes": b, "flops": f}


def tolerance(case):
    c = case
    if c["mode"] == "cpu":
        return "exact"  # bit for bit the CPU backend's arithmetic order
    if c["mode"] == "int8":
        # A chained activation next to a rounding tie takes another int8 value when the sums before it are
        # added in another order.
        return {"rel": 2e-2, "max": 0.3, "differ": 0.0} if c["kind"] == "model" else \
            {"rel": 2e-3, "max": 0.05, "differ": 0.0}
    if c["kind"] == "model":
        # The cache stores f16: its roundings alone put the logits 3.4e-4 from the 64-bit result, and a sum in
        # another order rounds a few keys and values to the other neighbour.
        return {"rel": 2e-4, "max": 2e-3, "differ": 0.0}
    return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}


# ---- the same results in 64 bits ----

def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _attn64(q, k, v, heads, kv_heads, hd):
    """Causal GQA attention of q's rows, the last of k's positions."""
    T, N = q.shape[0], k.shape[0]
    out = torch.empty(T, heads * hd, dtype=torch.float64, device=q.device)
    mask = torch.arange(N, device=q.device)[None, :] > torch.arange(N - T, N, device=q.device)[:, None]
    for h in range(heads):
        kv = h // (heads // kv_heads)
        s = q[:, h * hd:(h + 1) * hd] @ k[:, kv * hd:(kv + 1) * hd].t().contiguous() / math.sqrt(hd)
        out[:, h * hd:(h + 1) * hd] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[:, kv * hd:(kv + 1) * hd]
    return out


def _rope64(x, pos, heads, hd, theta):
    T = x.shape[0]
    f = theta ** (-torch.arange(0, hd, 2, device=x.device).double() / hd)
    a = torch.arange(pos, pos + T, device=x.device).double()[:, None, None] * f
    p = x.view(T, heads, hd // 2, 2)
    c, s = torch.cos(a), torch.sin(a)
    return torch.stack([p[..., 0] * c - p[..., 1] * s, p[..., 0] * s + p[..., 1] * c], -1).reshape(T, heads * hd)


def _host(d):
    return {k: v.cpu().numpy() for k, v in d.items()}


def _exact_linears(c, seed):
    shapes, blks, a = _linears_inputs(c, seed)

    def mul(k, x):
        dt, r, n = shapes[k]
        return x @ _dequant(blks[k], dt, r, n).t().contiguous()

    x = a["x"].double()
    n1 = _rms64(x, a["w1"])
    out = {k: mul(k, n1) for k in ("q", "k", "v")}
    out["proj"] = mul("o", a["att"].double())
    s = x + out["proj"]
    n2 = _rms64(s, a["w2"])
    out["ffn"] = mul("down", torch.nn.functional.silu(mul("gate", n2)) * mul("up", n2))
    out["out"] = s + out["ffn"]
    return _host(out)


def _exact_model(c, seed):
    geom, dtypes, toks, tensors = _model_inputs(c, seed)
    t = {n: (dt, sh, v) for n, dt, sh, v in tensors}
    heads, kvh, E = geom["n_heads"], geom["n_kv_heads"], geom["n_embd"]
    hd = E // heads

    def mat(name):
        dt, sh, v = t[name]
        return v.double() if dt == GGML_F32 else _dequant(v, dt, *sh)

    ids = torch.from_numpy(toks[:c["tokens"] + (c["step"] == "decode")].astype(np.int64)).cuda()
    x = mat("token_embd.weight")[ids]
    for i in range(geom["n_layers"]):
        p = f"blk.{i}."
        n = _rms64(x, t[p + "attn_norm.weight"][2])
        q, k, v = (n @ mat(p + f"attn_{j}.weight").t().contiguous() for j in "qkv")
        q = _rope64(q, 0, heads, hd, geom["rope_theta"])
        k = _rope64(k, 0, kvh, hd, geom["rope_theta"])
        x = x + _attn64(q, k, v, heads, kvh, hd) @ mat(p + "attn_output.weight").t().contiguous()
        n = _rms64(x, t[p + "ffn_norm.weight"][2])
        a = torch.nn.functional.silu(n @ mat(p + "ffn_gate.weight").t().contiguous())
        x = x + (a * (n @ mat(p + "ffn_up.weight").t().contiguous())) @ mat(p + "ffn_down.weight").t().contiguous()
    n = _rms64(x[-1:], t["output_norm.weight"][2])
    return {"logits": (n @ mat("output.weight").t().contiguous())[0].cpu().numpy()}


def exact(case, seed):
    c = case
    if c["kind"] == "linears":
        return _exact_linears(c, seed)
    if c["kind"] == "attn":
        q, k, v = (t.double() for t in _attn_inputs(c, seed))
        return _host({"o": _attn64(q, k, v, c["heads"], c["kv_heads"], c["head_dim"])})
    if c["kind"] == "head":
        dt, blk, x, w = _head_inputs(c, seed)
        n, rows = _rms64(x.double(), w), []
        for r in range(0, c["vocab"], 16384):  # in pieces: the whole table is large in 64 bits
            m = min(16384, c["vocab"] - r)
            per = blk.shape[0] // c["vocab"]
            rows.append(n @ _dequant(blk[r * per:(r + m) * per], dt, m, c["embd"]).t().contiguous())
        return [_host({"logits": torch.cat(rows, 1)}), [None] * c["tokens"]]
    return _exact_model(c, seed)
