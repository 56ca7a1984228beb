"""What this framework is used for, as a list of measurable cases: the smallest and largest
matrix-vector products of a decode step, short and long batches of columns, prompt MLPs, attention
over a long cache, decoder steps and layers through the ggml backend, and whole model calls.

Shapes are the repository's own (the Llama-3.2-3B and Qwen3-8B configurations of bench.py). Weights are
N(0, 0.02) in ggml's Q4_K / Q6_K blocks, activations N(0, 1), norm weights near 1. Everything a case
needs is made here from its seed with torch, so `exact` can form the same weights in 64 bits without
the library."""
import ctypes as C
import math

import numpy as np
import torch

import kernelcore_amd as kc
from kernelcore_amd import ggml_graph as gg

LLAMA_3B = dict(n_layer=28, n_embd=3072, n_head=24, n_head_kv=8, head_dim=128, n_ff=8192, n_vocab=128256,
                norm_eps=1e-5, rope_theta=500000.0, rope_neox=0, qk_norm=0, max_ctx=1024, max_batch=512)
QWEN3_8B = dict(n_layer=36, n_embd=4096, n_head=32, n_head_kv=8, head_dim=128, n_ff=12288, n_vocab=151936,
                norm_eps=1e-6, rope_theta=1000000.0, rope_neox=1, qk_norm=1, max_ctx=1536, max_batch=1024)
ARCH = {"3b": LLAMA_3B, "8b": QWEN3_8B}
BLOCK = {"q4k": 144, "q6k": 210}
# a layer's matrices: (name, tensor id, type of a Q4_K_M file)
MATRICES = (("wq", 4, "q4k"), ("wk", 5, "q4k"), ("wv", 6, "q6k"), ("wo", 7, "q4k"), ("wg", 9, "q4k"), ("wu", 10, "q4k"),
            ("wd", 11, "q6k"))


# ---- the cases ------------------------------------------------------------------------------------

def listed():
    return [
        # one projection of a decode step, called by name: the smallest call, latency counts
        dict(name="matvec_q4k_3072", kind="matvec", qtype="q4k", rows=3072, k=3072),
        # the output head of every decoded token: the largest matrix, streamed once
        dict(name="matvec_q6k_head", kind="matvec", qtype="q6k", rows=128256, k=3072),
        # a gate projection for a few tokens at once (drafted tokens, a handful of sequences)
        dict(name="matmul_q4k_cols12", kind="matmul", qtype="q4k", rows=8192, k=3072, cols=12),
        # a down projection for a short, ragged prompt
        dict(name="matmul_q6k_cols37", kind="matmul", qtype="q6k", rows=3072, k=8192, cols=37),
        # the MLP of a 512-token prompt, called by name
        dict(name="mlp_prompt_512", kind="mlp", embd=3072, ff=8192, down="q4k", cols=512),
        # an F16 value projection (files that keep attn_v in F16) for a ragged prompt
        dict(name="matmul_f16_cols77", kind="f16", rows=1024, k=4096, cols=77),
        # one token's attention over a long context
        dict(name="flash_decode_8k", kind="flash", heads=32, heads_kv=8, dim=128, tokens=1, ctx=8192),
        # a decode step as a llama.cpp build runs it: graph_compute over a stack of layers and the head
        dict(name="backend_decode_3b", kind="decoder", arch="3b", layers=8, past=575),
        # a layer of a 1024-token prompt through the backend
        dict(name="backend_prompt_8b_1024", kind="layer", arch="8b", tokens=1024, past=0),
        # a layer of a later, ragged chunk of a conversation (cache behind it) through the backend
        dict(name="backend_chunk_3b_200", kind="layer", arch="3b", tokens=200, past=1000),
        # a chat turn on the model driver: a short prompt, then decode steps sampled by the host (fewer
        # layers than the checkpoint's 28, here and below: a rounding of the 8-bit activations travels
        # through every layer after it, and the logits of all 28 would compare little but that)
        dict(name="model_turn_3b", kind="model", arch="3b", layers=16, prompt=48, steps=8),
        # a long prompt on the model driver
        dict(name="model_prompt_3b_512", kind="model", arch="3b", layers=12, prompt=512, steps=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matmul", "matmul", "mlp", "f16", "flash", "decoder", "layer", "layer", "model"])
    qtype = rng.choice(["q4k", "q6k"])
    if kind == "matvec":
        return dict(kind=kind, qtype=qtype, rows=8 * _log(rng, 32, 16032), k=256 * _log(rng, 2, 48))
    if kind == "matmul":
        return dict(kind=kind, qtype=qtype, rows=8 * _log(rng, 64, 2048), k=256 * _log(rng, 4, 48), cols=_log(rng, 2, 512))
    if kind == "mlp":
        return dict(kind=kind, embd=256 * rng.randint(4, 16), ff=256 * rng.randint(8, 48), down=qtype, cols=_log(rng, 9, 512))
    if kind == "f16":
        return dict(kind=kind, rows=8 * _log(rng, 32, 1024), k=8 * _log(rng, 64, 1024), cols=_log(rng, 1, 512))
    if kind == "flash":
        h = rng.choice([24, 32])
        return dict(kind=kind, heads=h, heads_kv=8, dim=rng.choice([64, 128]), tokens=rng.choice([1, 1, 1, 2, 5, 8]),
                    ctx=_log(rng, 64, 16384))
    arch = rng.choice(["3b", "8b"])
    if kind == "decoder":
        return dict(kind=kind, arch=arch, layers=rng.randint(2, 8), past=_log(rng, 8, 2000))
    if kind == "layer":
        return dict(kind=kind, arch=arch, tokens=_log(rng, 2, 1024), past=rng.choice([0, _log(rng, 8, 1000)]))
    return dict(kind=kind, arch="3b", layers=rng.randint(4, 12), prompt=_log(rng, 2, 512), steps=rng.randint(0, 6))


# ---- inputs (torch, from the seed alone) ----------------------------------------------------------

def _normal(seed, *shape):
    g = torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFFFFFF)
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _sub(seed, *ids):
    for i in ids:
        seed = (seed * 1000003 + i + 7) & 0x7FFFFFFFFFFF
    return seed


def _bytes(h):
    return h.contiguous().view(torch.uint8)


def _blocks(qtype, rows, k, seed):
    """rows x k weights N(0, 0.02) as ggml blocks: uint8 [rows, k / 256, block bytes]."""
    n = k // 256
    out = torch.empty(rows, n, BLOCK[qtype], dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 27) // k)
    for i, r0 in enumerate(range(0, rows, step)):
        r1 = min(rows, r0 + step)
        w = _normal(_sub(seed, i), r1 - r0, n, 256) * 0.02
        (_pack_q4k if qtype == "q4k" else _pack_q6k)(w, out[r0:r1])
    return out


def _pack_q4k(w, out):
    r, n, _ = w.shape
    w = w.view(r, n, 8, 32)
    lo = w.amin(-1).clamp(max=0.0)
    sc = ((w.amax(-1) - lo) / 15).clamp(min=1e-9)
    d = (sc.amax(-1, keepdim=True) / 63).half()
    m = (-lo.amin(-1, keepdim=True) / 63).half()
    ls = (sc / d.float()).round().clamp(1, 63)
    lm = (-lo / m.float().clamp(min=1e-9)).round().clamp(0, 63)
    q = ((w + (m.float() * lm)[..., None]) / (d.float() * ls)[..., None]).round().clamp(0, 15).to(torch.uint8)
    ls, lm = ls.to(torch.uint8), lm.to(torch.uint8)
    out[..., 0:2], out[..., 2:4] = _bytes(d), _bytes(m)
    out[..., 4:8] = ls[..., :4] | ((ls[..., 4:] >> 4) << 6)
    out[..., 8:12] = lm[..., :4] | ((lm[..., 4:] >> 4) << 6)
    out[..., 12:16] = (ls[..., 4:] & 15) | ((lm[..., 4:] & 15) << 4)
    out[..., 16:] = (q[:, :, 0::2] | (q[:, :, 1::2] << 4)).reshape(r, n, 128)


def _pack_q6k(w, out):
    r, n, _ = w.shape
    w = w.view(r, n, 16, 16)
    sc = (w.abs().amax(-1) / 31).clamp(min=1e-9)
    d = (sc.amax(-1, keepdim=True) / 127).half()
    ls = (sc / d.float()).round().clamp(1, 127)
    q = ((w / (d.float() * ls)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8).view(r, n, 2, 4, 32)
    ql = torch.stack([(q[:, :, :, a] & 15) | ((q[:, :, :, a + 2] & 15) << 4) for a in (0, 1)], 3)
    qh = sum((q[:, :, :, a] >> 4) << (2 * a) for a in range(4))
    out[..., :128], out[..., 128:192] = ql.reshape(r, n, 128), qh.reshape(r, n, 64)
    out[..., 192:208], out[..., 208:210] = ls.to(torch.uint8), _bytes(d)


def _dims(arch, name):
    c = ARCH[arch]
    E, Q, KV, F = c["n_embd"], c["n_head"] * c["head_dim"], c["n_head_kv"] * c["head_dim"], c["n_ff"]
    return dict(wq=(Q, E), wk=(KV, E), wv=(KV, E), wo=(E, Q), wg=(F, E), wu=(F, E), wd=(E, F))[name]


def _norm_weight(n, seed):
    return 1.0 + 0.1 * (2.0 * torch.rand(n, generator=torch.Generator().manual_seed(seed & 0x7FFFFFFFFFFF)) - 1.0)


def _tokens(case, seed):
    r = np.random.default_rng(seed)
    return r.integers(0, ARCH[case["arch"]]["n_vocab"], case["prompt"] + case["steps"]).astype(np.int32)


def _cache_rows(case, seed, which, layer):
    """The cache rows of the positions before this step (fp16, as set_rows stores them)."""
    c = ARCH[case["arch"]]
    return _normal(_sub(seed, 500 + which, layer), case["past"], c["n_head_kv"] * c["head_dim"]).half()


# ---- memory and handles ---------------------------------------------------------------------------

class _View:
    """A kcMalloc allocation as torch reads it (the __cuda_array_interface__ of its bytes)."""

    def __init__(self, buf, ptr, shape, dtype):
        self.buf = buf
        t = {torch.float32: "<f4", torch.float16: "<f2", torch.int32: "<i4", torch.uint8: "|u1", torch.int64: "<i8"}[dtype]
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": t, "data": (ptr, False), "version": 2}


def _as_torch(buf, shape, dtype=torch.float32, ptr=None):
    return torch.as_tensor(_View(buf, ptr or buf.ptr, shape, dtype), device="cuda")


class _Buffer(kc.Buffer):
    """A kcMalloc allocation freed with the last state, view or tensor that holds it."""

    def __del__(self):
        self.free()


class _State(dict):
    """What a case keeps between calls."""

    def buffer(self, nbytes):
        b = _Buffer(nbytes)
        self.setdefault("buffers", []).append(b)
        return b

    def put(self, t):
        """A device copy of a torch tensor in the library's memory."""
        t = t.contiguous().cuda()
        b = self.buffer(t.numel() * t.element_size())
        _as_torch(b, t.shape, t.dtype).copy_(t)
        return b

    def zeros(self, nbytes):
        b = self.buffer(nbytes)
        _as_torch(b, (b.nbytes,), torch.uint8).zero_()
        return b

    def weights(self, qtype, rows, k, seed):
        """A weight stream of the library (repacked once, as a program does when it loads a model)."""
        b = self.buffer(kc.stream_bytes(qtype, rows, k))
        _repack(qtype, rows, k, seed, b.ptr)
        return b

    def __del__(self):
        kc.synchronize()
        for n in ("backend", "model"):
            if n in self:
                self[n].close()


def _repack(qtype, rows, k, seed, dst):
    blocks = _blocks(qtype, rows, k, seed)
    raw = _Buffer(blocks.numel())
    _as_torch(raw, blocks.shape, torch.uint8).copy_(blocks)
    torch.cuda.synchronize()
    kc.launch("repack_kquant", kc.KquantRepackArgs(raw.ptr, dst, kc.QTYPE[qtype], rows, k))


_STREAM = []


def _stream():
    if not _STREAM:
        kc.init()
        s = C.c_void_p()
        kc.call("kcStreamCreate", C.byref(s))
        _STREAM.append(s)
    return _STREAM[0]


def prepare(case, seed):
    s = _State(case=case, stream=_stream())
    globals()["_prepare_" + case["kind"]](s, case, seed)
    torch.cuda.synchronize()
    return s


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _launches(s):
    for name, args in s["launches"]:
        kc.launch(name, args, s["stream"])
    return s["out"]


# one activation vector quantized and multiplied
def _prepare_matvec(s, c, seed):
    rows, k = c["rows"], c["k"]
    w, x = s.weights(c["qtype"], rows, k, _sub(seed, 1)), s.put(_normal(_sub(seed, 2), k))
    slot, y = s.zeros(k // 32 * 40), s.zeros(4 * rows)
    s["launches"] = [("quantize_q8x4", kc.QuantizeArgs(x.ptr, slot.ptr, slot.ptr + k, k // 32)),
                     ("matvec_%s_q8" % c["qtype"], kc.MatvecQ4Q8Args(w.ptr, slot.ptr, slot.ptr + k, y.ptr, None, rows, k))]
    s["out"] = _as_torch(y, (rows,))


_run_matvec = _launches


def _matmul(qtype, w, slots, y, rows, k, cols):
    return ("matmul_%s_q8kx%d" % (qtype, 8 if cols >= 8 else 4), kc.MatmulKQ8Args(w.ptr, slots.ptr, y.ptr, None, rows, k, cols, 8))


# a batch of activation columns quantized and multiplied
def _prepare_matmul(s, c, seed):
    rows, k, n = c["rows"], c["k"], c["cols"]
    w, x = s.weights(c["qtype"], rows, k, _sub(seed, 1)), s.put(_normal(_sub(seed, 2), n, k))
    slots, y = s.zeros(n * k // 256 * 340), s.zeros(4 * rows * n)
    s["launches"] = [("quantize_cols_k", kc.QuantizeColsArgs(x.ptr, slots.ptr, None, k, n)),
                     _matmul(c["qtype"], w, slots, y, rows, k, n)]
    s["out"] = _as_torch(y, (n, rows))


_run_matmul = _launches


# quantize, gate and up, SwiGLU with its quantization, down
def _prepare_mlp(s, c, seed):
    E, F, n = c["embd"], c["ff"], c["cols"]
    wg, wu = s.weights("q4k", F, E, _sub(seed, 1)), s.weights("q4k", F, E, _sub(seed, 2))
    wd, x = s.weights(c["down"], E, F, _sub(seed, 3)), s.put(_normal(_sub(seed, 4), n, E))
    g, u, act, y = s.zeros(4 * F * n), s.zeros(4 * F * n), s.zeros(4 * F * n), s.zeros(4 * E * n)
    se, sf = s.zeros(n * E // 256 * 340), s.zeros(n * F // 256 * 340)
    s["launches"] = [("quantize_cols_k", kc.QuantizeColsArgs(x.ptr, se.ptr, None, E, n)),
                     _matmul("q4k", wg, se, g, F, E, n), _matmul("q4k", wu, se, u, F, E, n),
                     ("silu_mul_q8kf", kc.SiluMulQ8FArgs(g.ptr, u.ptr, act.ptr, sf.ptr, None, F, n)),
                     _matmul(c["down"], wd, sf, y, E, F, n)]
    s["out"] = _as_torch(y, (n, E))


_run_mlp = _launches


# fp16 weights times f32 activations
def _prepare_f16(s, c, seed):
    rows, k, n = c["rows"], c["k"], c["cols"]
    w = s.put((_normal(_sub(seed, 1), rows, k) * 0.02).half())
    x, y = s.put(_normal(_sub(seed, 2), n, k)), s.zeros(4 * rows * n)
    s["launches"] = [("matmul_f16", kc.MatmulF16Args(w.ptr, x.ptr, y.ptr, None, rows, k, n))]
    s["out"] = _as_torch(y, (n, rows))


_run_f16 = _launches


# attention of a few query tokens over a cache in ggml's layout [position][kv head][dim]
def _flash_inputs(c, seed):
    H, K, D, N, T = c["heads"], c["heads_kv"], c["dim"], c["tokens"], c["ctx"]
    q = _normal(_sub(seed, 1), N, H, D)
    k, v = _normal(_sub(seed, 2), T, K, D).half(), _normal(_sub(seed, 3), T, K, D).half()
    tp = (T + 7) // 8 * 8
    at = torch.arange(tp, device="cuda")[None] <= torch.arange(T - N, T, device="cuda")[:, None]
    mask = torch.where(at, 0.0, -math.inf).half()
    return q, k, v, mask, tp


def _prepare_flash(s, c, seed):
    H, K, D, N, T = c["heads"], c["heads_kv"], c["dim"], c["tokens"], c["ctx"]
    q, k, v, mask, tp = _flash_inputs(c, seed)
    bq, bk, bv, bm = s.put(q), s.put(k), s.put(v), s.put(mask)
    out, part = s.zeros(4 * N * H * D), s.zeros(4 * N * H * ((T + 63) // 64) * (D + 2))
    d = kc.FaDims(H=H, T=T, D=D, group=H // K, tp=tp, k_row=K * D // 2, k_head=D // 2, v_row=K * D // 2, v_head=D // 2,
                  N=N, q_tok=H * D, q_head=D, m_row=tp // 2, has_mask=int(N > 1), H_kv=K)
    s["launches"] = [("flash_decode_f16", kc.FlashDecodeArgs(bq.ptr, bk.ptr, bv.ptr, bm.ptr, out.ptr, part.ptr, None, d,
                                                             1.0 / math.sqrt(D)))]
    s["out"] = _as_torch(out, (N, H, D))


_run_flash = _launches


# ---- the ggml backend: llama.cpp's graphs over tensors the program owns ----------------------------

def _graph(s, c, seed, tokens, layers):
    """The graph's memory: weights by layer, caches holding the past positions, the step's inputs."""
    cfg = ARCH[c["arch"]]
    past = c["past"]
    n_kv = (past + tokens + 255) // 256 * 256
    shape = gg.LayerShape.of_model(cfg, n_kv)
    held = {}

    def alloc(nbytes, type_, ne):
        b = s.buffer(kc.stream_bytes(type_, ne[1], ne[0]) if type_ in ("q4k", "q6k") else nbytes)
        held[b.ptr] = b
        return b.ptr

    g = gg.Graph(alloc)
    if layers:
        io, w, ts, out = gg.decoder(g, shape, layers, tokens, n_kv)
        per_layer = w["layers"]
    else:
        out = t = gg.llama_layer(g, shape, tokens, n_kv)
        io, w, per_layer, out = t, {}, [t], t["out"]

    def fill(t, v):
        _as_torch(held[t.data], v.shape, v.dtype).copy_(v)

    def matrix(t, qtype, rows, k, sd):
        _repack(qtype, rows, k, sd, t.data)

    kv = cfg["n_head_kv"] * cfg["head_dim"]
    caches = []
    for l, lw in enumerate(per_layer):
        for name, tid, qtype in MATRICES:
            matrix(lw[name], qtype, *_dims(c["arch"], name), _sub(seed, tid, l))
        norms = [("attn_norm", 3, cfg["n_embd"]), ("ffn_norm", 8, cfg["n_embd"])]
        if cfg["qk_norm"]:
            norms += [("q_norm", 12, cfg["head_dim"]), ("k_norm", 13, cfg["head_dim"])]
        for name, tid, n in norms:
            fill(lw[name], _norm_weight(n, _sub(seed, tid, l)))
        for which, name in enumerate(("k_cache", "v_cache")):
            full = torch.zeros(n_kv, kv, dtype=torch.float16, device="cuda")
            full[:past] = _cache_rows(c, seed, which, l)
            fill(lw[name], full)
            caches.append(_as_torch(held[lw[name].data], (tokens, kv), torch.float16, lw[name].data + past * kv * 2))
    if layers:
        fill(w["output_norm"], _norm_weight(cfg["n_embd"], _sub(seed, 1, 0)))
        matrix(w["output"], "q6k", cfg["n_vocab"], cfg["n_embd"], _sub(seed, 2, 0))
    fill(io["x"], _normal(_sub(seed, 600), tokens, cfg["n_embd"]))
    pos = torch.arange(past, past + tokens, dtype=torch.int32)
    at = torch.arange(io["mask"].ne[0])[None] <= pos[:, None]
    s["inputs"] = [(held[io[n].data], v.numpy()) for n, v in
                   (("pos", pos), ("kv_idx", pos.long()), ("mask", torch.where(at, 0.0, -math.inf).half()))]
    torch.cuda.synchronize()
    s["backend"] = kc.GgmlBackend(attn_tokens=max(8, tokens))
    s["graph"], s["nodes"] = g, kc.GgmlNodes(g.nodes)
    n_out = cfg["n_vocab"] if layers else cfg["n_embd"]
    s["out"] = [_as_torch(held[out.data], (1 if layers else tokens, n_out))] + caches


def _compute(s):
    """One step: the host hands over its inputs (positions, cache rows, the mask), then computes the graph."""
    for buf, a in s["inputs"]:
        buf.upload(a)
    s["backend"].compute(s["nodes"])
    return s["out"]


def _prepare_decoder(s, c, seed):
    _graph(s, c, seed, 1, c["layers"])


def _prepare_layer(s, c, seed):
    _graph(s, c, seed, c["tokens"], 0)


_run_decoder = _run_layer = _compute


# ---- the model driver -----------------------------------------------------------------------------

def _prepare_model(s, c, seed):
    cfg = dict(ARCH[c["arch"]], n_layer=c["layers"])
    s["tokens"] = _tokens(c, _sub(seed, 700))
    m = s["model"] = kc.Model(**cfg)
    E, V = cfg["n_embd"], cfg["n_vocab"]
    m.set_tensor("token_embd", -1, _blocks("q4k", V, E, _sub(seed, 0, 0)).cpu().numpy())
    m.set_tensor("output_norm", -1, _norm_weight(E, _sub(seed, 1, 0)).numpy())
    m.set_tensor("output", -1, _blocks("q6k", V, E, _sub(seed, 2, 0)).cpu().numpy())
    for l in range(cfg["n_layer"]):
        for name, tid, qtype in MATRICES:
            m.set_tensor(tid, l, _blocks(qtype, *_dims(c["arch"], name), _sub(seed, tid, l)).cpu().numpy())
        m.set_tensor("attn_norm", l, _norm_weight(E, _sub(seed, 3, l)).numpy())
        m.set_tensor("ffn_norm", l, _norm_weight(E, _sub(seed, 8, l)).numpy())


def _run_model(s):
    m, n = s["model"], s["case"]["prompt"]
    m.reset()
    out = [m.forward(s["tokens"][:n])]
    for t in s["tokens"][n:]:  # the host picks each next token
        out.append(m.forward(np.array([t], np.int32)))
    return out


# ---- what a pass cannot do without -----------------------------------------------------------------

def _mat(qtype, rows, k, cols):
    return rows * (k // 256) * BLOCK[qtype], 2 * rows * k * cols


def _layer_work(arch, n, ctx):
    c = ARCH[arch]
    b = f = 0
    for name, _, qtype in MATRICES:
        mb, mf = _mat(qtype, *_dims(arch, name), n)
        b, f = b + mb, f + mf
    kv = c["n_head_kv"] * c["head_dim"]
    b += 2 * 2 * kv * (ctx + n)
    seen = n * ctx + n * (n + 1) // 2
    return b, f + 4 * seen * c["n_head"] * c["head_dim"]


def work(case):
    c, kind = case, case["kind"]
    if kind in ("matvec", "matmul"):
        n = c.get("cols", 1)
        b, f = _mat(c["qtype"], c["rows"], c["k"], n)
        return {"bytes": b + 4 * n * (c["k"] + c["rows"]), "flops": f}
    if kind == "mlp":
        b1, f1 = _mat("q4k", c["ff"], c["embd"], c["cols"])
        b2, f2 = _mat(c["down"], c["embd"], c["ff"], c["cols"])
        return {"bytes": 2 * b1 + b2 + 8 * c["cols"] * c["embd"], "flops": 2 * f1 + f2}
    if kind == "f16":
        return {"bytes": 2 * c["rows"] * c["k"] + 4 * c["cols"] * (c["rows"] + c["k"]), "flops": 2 * c["rows"] * c["k"] * c["cols"]}
    if kind == "flash":
        n = c["tokens"] * c["heads"] * c["dim"]
        return {"bytes": 4 * c["ctx"] * c["heads_kv"] * c["dim"] + 8 * n, "flops": 4 * n * c["ctx"]}
    cfg = ARCH[c["arch"]]
    hb, hf = _mat("q6k", cfg["n_vocab"], cfg["n_embd"], 1)
    if kind == "decoder":
        b, f = _layer_work(c["arch"], 1, c["past"])
        return {"bytes": c["layers"] * b + hb, "flops": c["layers"] * f + hf}
    if kind == "layer":
        b, f = _layer_work(c["arch"], c["tokens"], c["past"])
        return {"bytes": b + 8 * c["tokens"] * cfg["n_embd"], "flops": f}
    b = f = 0
    for n, past in [(c["prompt"], 0)] + [(1, c["prompt"] + i) for i in range(c["steps"])]:
        lb, lf = _layer_work(c["arch"], n, past)
        b, f = b + c["layers"] * lb + hb, f + c["layers"] * lf + hf
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the distance from `exact` measured for each kind: 32-bit sums of exact integer
    products (2e-7), of fp16 weights times activations split in two fp16 parts (6e-7), online softmax
    (3e-7); where a product's activations are rounded to 8 bits from another product's sums, a value at
    a rounding tie moves by a step (an MLP 4e-4, a layer 7e-3 after its three roundings, 8 layers and the head
    3e-2, 16 layers 6e-2)."""
    return {"rel": {"matvec": 1e-6, "matmul": 1e-6, "f16": 2.5e-6, "flash": 1.5e-6, "mlp": 2e-3, "layer": 0.03,
                    "decoder": 0.1, "model": 0.25}[case["kind"]]}


# ---- the same in 64 bits ----------------------------------------------------------------------------

def _unpack_q4k(b):
    d, m = (b[..., i:i + 2].contiguous().view(torch.float16).double() for i in (0, 2))
    s = b[..., 4:16]
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
    q = b[..., 16:].reshape(*b.shape[:2], 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 3).reshape(*b.shape[:2], 8, 32)
    return (q.double() * (d * sc.double())[..., None] - (m * mn.double())[..., None]).view(b.shape[0], -1)


def _weights64(qtype, rows, k, seed):
    b = _blocks(qtype, rows, k, seed)
    if qtype == "q4k":
        return _unpack_q4k(b)
    n = k // 256
    d = b[..., 208:210].contiguous().view(torch.float16).double()
    sc = b[..., 192:208].contiguous().view(torch.int8).double()
    ql, qh = b[..., :128].view(rows, n, 2, 2, 32), b[..., 128:192].view(rows, n, 2, 32)
    q = torch.stack([((ql[:, :, :, a & 1] >> (4 * (a >> 1))) & 15) | (((qh >> (2 * a)) & 3) << 4) for a in range(4)], 3)
    return ((q.double() - 32).view(rows, n, 16, 16) * (d * sc)[..., None]).view(rows, k)


def _q8(x, n):
    """Activations rounded to 8 bits in groups of n values, as the path defines them."""
    v = x.view(*x.shape[:-1], -1, n)
    d = v.float().abs().amax(-1, keepdim=True) / 127
    inv = torch.where(d > 0, 1 / d, torch.zeros_like(d)).double()
    t = v * inv
    q = torch.trunc(t + torch.where(t >= 0, 0.5, -0.5)).clamp(-127, 127)
    return (q * d.double()).reshape(x.shape)


def _rms64(x, w, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w.double().cuda()


def _rope64(x, pos, cfg):
    D = cfg["head_dim"]
    th = pos.double()[:, None] * cfg["rope_theta"] ** (-2.0 * torch.arange(D // 2, device="cuda").double() / D)
    c, s = torch.cos(th)[:, None], torch.sin(th)[:, None]
    y = torch.empty_like(x)
    a, b = (slice(0, D // 2), slice(D // 2, D)) if cfg["rope_neox"] else (slice(0, D, 2), slice(1, D, 2))
    y[..., a], y[..., b] = x[..., a] * c - x[..., b] * s, x[..., a] * s + x[..., b] * c
    return y


def _attend64(q, k, v, group, first):
    """q [N, H, D] over k, v [T, Hkv, D]; query i sees the positions up to first + i."""
    N, H, D = q.shape
    out = torch.empty_like(q)
    hide = torch.arange(k.shape[0], device="cuda")[None] > first + torch.arange(N, device="cuda")[:, None]
    for h in range(H):
        kh, vh = k[:, h // group].contiguous(), v[:, h // group].contiguous()
        s = (q[:, h].contiguous() @ kh.t().contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(hide, -math.inf), -1) @ vh
    return out


def _layer64(arch, x, l, seed, past, kc_, vc_, last=False):
    """One layer on x [N, embd] after `past` cached positions (kc_, vc_: the caches so far, fp16 values in
    64 bits): the new x and caches. A batch rounds activations per 256 values, a single token per 32; `last`:
    the last layer of a prompt continues with its last token alone."""
    cfg = ARCH[arch]
    n, D = x.shape[0], cfg["head_dim"]
    w = lambda name, a, g: _q8(a, g) @ _weights64(dict((m[0], m[2]) for m in MATRICES)[name], *_dims(arch, name),  # noqa: E731
                                                  _sub(seed, dict((m[0], m[1]) for m in MATRICES)[name], l)).t()
    g = 256 if n > 1 else 32
    h = _rms64(x, _norm_weight(cfg["n_embd"], _sub(seed, 3, l)), cfg["norm_eps"])
    q, k, v = w("wq", h, g).view(n, -1, D), w("wk", h, g).view(n, -1, D), w("wv", h, g).view(n, -1, D)
    if cfg["qk_norm"]:
        q = _rms64(q, _norm_weight(D, _sub(seed, 12, l)), cfg["norm_eps"])
        k = _rms64(k, _norm_weight(D, _sub(seed, 13, l)), cfg["norm_eps"])
    pos = torch.arange(past, past + n, device="cuda")
    q, k = _rope64(q, pos, cfg), _rope64(k, pos, cfg)
    kc_, vc_ = torch.cat([kc_, k.half().double()]), torch.cat([vc_, v.half().double()])
    o = w("wo", _attend64(q, kc_, vc_, cfg["n_head"] // cfg["n_head_kv"], past).reshape(n, -1), g)
    x = x + o
    if last:
        x, g = x[-1:], 32
    h = _rms64(x, _norm_weight(cfg["n_embd"], _sub(seed, 8, l)), cfg["norm_eps"])
    a, u = w("wg", h, g), w("wu", h, g)
    return x + w("wd", a / (1 + torch.exp(-a)) * u, g), kc_, vc_


def _head64(arch, x, seed):
    cfg = ARCH[arch]
    h = _rms64(x[-1:], _norm_weight(cfg["n_embd"], _sub(seed, 1, 0)), cfg["norm_eps"])
    return _q8(h, 32) @ _weights64("q6k", cfg["n_vocab"], cfg["n_embd"], _sub(seed, 2, 0)).t()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("matvec", "matmul"):
        x = _normal(_sub(seed, 2), *([c["cols"]] if kind == "matmul" else []), c["k"]).double()
        return _q8(x, 256 if kind == "matmul" else 32) @ _weights64(c["qtype"], c["rows"], c["k"], _sub(seed, 1)).t()
    if kind == "mlp":
        x = _q8(_normal(_sub(seed, 4), c["cols"], c["embd"]).double(), 256)
        a, u = (x @ _weights64("q4k", c["ff"], c["embd"], _sub(seed, i)).t() for i in (1, 2))
        return _q8(a / (1 + torch.exp(-a)) * u, 256) @ _weights64(c["down"], c["embd"], c["ff"], _sub(seed, 3)).t()
    if kind == "f16":
        w = (_normal(_sub(seed, 1), c["rows"], c["k"]) * 0.02).half().double()
        return _normal(_sub(seed, 2), c["cols"], c["k"]).double() @ w.t()
    if kind == "flash":
        q, k, v, _, _ = _flash_inputs(c, seed)
        return _attend64(q.double(), k.double(), v.double(), c["heads"] // c["heads_kv"], c["ctx"] - c["tokens"])
    cfg = ARCH[c["arch"]]
    heads = (-1, cfg["n_head_kv"], cfg["head_dim"])
    if kind in ("decoder", "layer"):
        n, past = c.get("tokens", 1), c["past"]
        x, rows = _normal(_sub(seed, 600), n, cfg["n_embd"]).double(), []
        for l in range(c.get("layers", 1)):
            x, k, v = _layer64(c["arch"], x, l, seed, past, *(_cache_rows(c, seed, i, l).double().view(heads) for i in (0, 1)))
            rows += [k[past:].reshape(n, -1), v[past:].reshape(n, -1)]
        return [x if kind == "layer" else _head64(c["arch"], x, seed)] + rows
    tokens = torch.from_numpy(_tokens(c, _sub(seed, 700))).long().cuda()
    embd = _blocks("q4k", cfg["n_vocab"], cfg["n_embd"], _sub(seed, 0, 0))
    cache = [[torch.zeros(0, *heads[1:], dtype=torch.float64, device="cuda")] * 2 for _ in range(c["layers"])]
    out, past = [], 0
    for step in [tokens[:c["prompt"]]] + [t[None] for t in tokens[c["prompt"]:]]:
        x = _unpack_q4k(embd[step])
        for l in range(c["layers"]):
            x, *cache[l] = _layer64(c["arch"], x, l, seed, past, *cache[l], last=len(step) > 1 and l + 1 == c["layers"])
        past += len(step)
        out.append(_head64(c["arch"], x, seed)[0])
    return out

