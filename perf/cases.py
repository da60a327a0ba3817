"""Performance cases: the work that a program on this framework has it do, at the sizes it does it.

Five kinds of work, each through the public C entry points that a program calls:

* ``proj``   one quantized matrix product (a projection, an output head) over T tokens
* ``attn``   a transformer layer's attention half: norm, QKV, (QK-Norm,) RoPE, KV append, attention
             over the cache, output projection, residual
* ``ffn``    the dense feed-forward half: norm, gate / up, SwiGLU, down, residual
* ``moe``    the routed feed-forward half: norm, router, top-k, expert products, weighted sum
* ``model``  a whole session step: token ids in, logits on the host out

The layer kinds queue their graph with ``ggml_backend_graph_compute_async``, as the decode loop
does; the model kind is ``Session.forward``, which returns when the logits are on the host. T = 1
is decoding, a few to a few dozen tokens a batched step or a short prompt, hundreds a prompt.
Outputs are the graph's own output tensors, seen in place, and the cache rows the step appended.

Shapes are those of the package's model configurations (``CONFIGS``). Weights are N(0, 0.02)
values quantized to each type's block format by a plain min / max quantizer.
"""
from __future__ import annotations

import ctypes as C
import importlib.util
import math
import os
import random
import sys
import tempfile
import zlib

import numpy as np
import torch  # first: the libraries below then share its HIP runtime

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
F64 = torch.float64


def _package():
    if "ggml_loader_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "ggml_loader_amd", os.path.join(ROOT, "ggml-loader_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["ggml_loader_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["ggml_loader_amd"]


gl = _package()
TYPES = {"q4_0": gl.Q4_0, "q8_0": gl.Q8_0, "q4_K": gl.Q4_K, "q5_K": gl.Q5_K, "q6_K": gl.Q6_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_K": (256, 144), "q5_K": (256, 176), "q6_K": (256, 210)}


# ---------------------------------------------------------------------------------------------
# the cases

# the attention geometry of the package's configurations
HEADS = {
    "llama": dict(embd=3072, head=24, head_kv=8, hd=128, neox=False, qk_norm=False, fused=False, base=5e5, eps=1e-5),
    "qwen3": dict(embd=2560, head=32, head_kv=8, hd=128, neox=True, qk_norm=True, fused=False, base=1e6, eps=1e-6),
    "phi3": dict(embd=3072, head=32, head_kv=32, hd=96, neox=True, qk_norm=False, fused=True, base=1e4, eps=1e-5),
    "qwen3moe": dict(embd=2048, head=32, head_kv=4, hd=128, neox=True, qk_norm=True, fused=False, base=1e6, eps=1e-6),
}


def listed():
    return [
        # one projection of one token: the smallest call, all latency
        dict(name="proj_q4_0_1", kind="proj", type="q4_0", K=4096, N=4096, T=1),
        # the output head of a Q4_K_M file: the largest matrix that every decoded token reads
        dict(name="head_q6_K_1", kind="proj", type="q6_K", K=2560, N=151936, T=1),
        # decoding one token deep in a context
        dict(name="attn_q4_K_decode8192", kind="attn", arch="qwen3", type="q4_K", past=8192, T=1),
        # a 16-token step (parallel sequences' drafts, a prompt's tail) in the middle of a context
        dict(name="attn_q4_K_step16_4096", kind="attn", arch="qwen3moe", type="q4_K", past=4096, T=16),
        # a prompt from an empty cache
        dict(name="attn_q8_0_prompt512", kind="attn", arch="phi3", type="q8_0", past=0, T=512),
        # a later chunk of a long prompt, ragged
        dict(name="attn_q4_K_chunk1000_3001", kind="attn", arch="qwen3", type="q4_K", past=3001, T=1000),
        # the feed-forward half of one decoded token
        dict(name="ffn_q4_K_1", kind="ffn", type="q4_K", embd=2560, ff=9728, T=1),
        # a short prompt
        dict(name="ffn_q4_0_prompt37", kind="ffn", type="q4_0", embd=3072, ff=8192, T=37),
        # an ordinary prompt
        dict(name="ffn_q4_K_prompt512", kind="ffn", type="q4_K", embd=2560, ff=9728, T=512),
        # routed experts: a 16-token step, and a prompt
        dict(name="moe_q4_K_step16", kind="moe", type="q4_K", embd=2048, ff=768, experts=128, k=8, T=16),
        dict(name="moe_q4_K_prompt384", kind="moe", type="q4_K", embd=2048, ff=768, experts=128, k=8, T=384),
        # whole decode steps of a model, logits on the host: eight of its layers, and its head
        dict(name="model_q4_0_decode2048", kind="model", arch="llama", type="q4_0", layers=8, ff=8192, vocab=128256,
             past=2048, T=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _drawn(rng):
    kind = rng.choice(("proj", "proj", "attn", "attn", "ffn", "ffn", "moe", "model"))
    wtype = rng.choice(tuple(TYPES))
    tokens = 1 if rng.random() < 0.35 else _log(rng, 2, 640)
    if kind == "proj":
        # rows from a key projection to an output head, odd counts among them
        rows = _log(rng, 512, 152000)
        return dict(kind=kind, type=wtype, K=256 * _log(rng, 4, 38), N=rows - rows % rng.choice((1, 2, 16, 64)),
                    T=tokens)
    if kind == "attn":
        past = 0 if tokens > 1 and rng.random() < 0.4 else _log(rng, 33, 8192)
        return dict(kind=kind, arch=rng.choice(tuple(HEADS)), type=wtype, past=past, T=tokens)
    if kind == "ffn":
        return dict(kind=kind, type=wtype, embd=256 * rng.randint(6, 16), ff=256 * rng.randint(12, 40), T=tokens)
    if kind == "moe":
        return dict(kind=kind, type=wtype, embd=256 * rng.randint(4, 10), ff=256 * rng.randint(2, 5),
                    experts=8 * rng.randint(2, 16), k=rng.randint(2, 8), T=tokens)
    return dict(kind=kind, arch=rng.choice(("llama", "qwen3")), type=wtype, layers=rng.randint(1, 3),
                ff=256 * rng.randint(16, 38), vocab=_log(rng, 4000, 32064), past=_log(rng, 16, 2048),
                T=min(tokens, 300))


def draw(rng: random.Random):
    most = [work(c) for c in listed()]
    flops, size = max(w["flops"] for w in most), max(w["bytes"] for w in most)
    while True:
        case = _drawn(rng)
        w = work(case)
        if w["flops"] <= flops and w["bytes"] <= size:
            return case


# ---------------------------------------------------------------------------------------------
# seeded values and block formats (bytes as in GGUF files)

def _gen(seed, name):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) << 32) + zlib.crc32(name.encode()))
    return g


def _randn(seed, name, *shape):
    return torch.randn(*shape, generator=_gen(seed, name), device=DEV)


def _half_bytes(x):
    return x.to(torch.float16).view(torch.uint8)


def _pack_sc_m(sc, mn):
    """The 6-bit scales and minimums of eight sub-blocks in 12 bytes."""
    lo = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    hi = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
    return torch.cat([lo, hi, (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1).to(torch.uint8)


def _quantize(x, wtype):
    """Rows x (multiples of a block long) as the type's blocks, and the values those blocks hold."""
    n = x.shape[0]
    qk, size = BLOCK[wtype]
    b = x.reshape(-1, qk)
    if wtype in ("q4_0", "q8_0"):
        big = b.gather(1, b.abs().argmax(1, keepdim=True))
        d = (big / -8 if wtype == "q4_0" else big.abs() / 127).to(torch.float16)
        inv = torch.where(d == 0, torch.zeros_like(big), 1 / d.float())
        if wtype == "q4_0":
            q = (b * inv + 8.5).floor().clamp(0, 15).to(torch.int32)
            raw = torch.cat([_half_bytes(d), (q[:, :16] | (q[:, 16:] << 4)).to(torch.uint8)], 1)
            val = (q - 8).float() * d.float()
        else:
            q = (b * inv).round().clamp(-127, 127)
            raw = torch.cat([_half_bytes(d), q.to(torch.int8).view(torch.uint8)], 1)
            val = q * d.float()
    elif wtype == "q6_K":
        s = b.reshape(-1, 16, 16)
        scale = s.abs().amax(2) / 31
        d = (scale.amax(1, keepdim=True) / 127).to(torch.float16)
        sc = (scale / d.float()).round().clamp(1, 127)
        step = (d.float() * sc)[:, :, None]
        q = ((s / step).round().clamp(-32, 31) + 32).to(torch.int32)
        val = (q - 32).float() * step
        h = q.reshape(-1, 2, 4, 32)          # half, group m, byte j
        ql = torch.cat([(h[:, :, 0] & 15) | ((h[:, :, 2] & 15) << 4), (h[:, :, 1] & 15) | ((h[:, :, 3] & 15) << 4)], 2)
        qh = (h[:, :, 0] >> 4) | ((h[:, :, 1] >> 4) << 2) | ((h[:, :, 2] >> 4) << 4) | ((h[:, :, 3] >> 4) << 6)
        raw = torch.cat([ql.reshape(-1, 128).to(torch.uint8), qh.reshape(-1, 64).to(torch.uint8),
                         sc.to(torch.int8).view(torch.uint8), _half_bytes(d)], 1)
    else:
        top = 15 if wtype == "q4_K" else 31
        s = b.reshape(-1, 8, 32)
        low = (-s.amin(2)).clamp(min=0)
        scale = (s.amax(2) + low) / top
        d, dm = ((v.amax(1, keepdim=True) / 63).to(torch.float16) for v in (scale, low))
        sc = (scale / d.float()).round().clamp(1, 63)
        mn = (low / dm.float()).round().clamp(0, 63)
        step, off = (d.float() * sc)[:, :, None], (dm.float() * mn)[:, :, None]
        q = ((s + off) / step).round().clamp(0, top).to(torch.int32)
        val = q.float() * step - off
        q = q.reshape(-1, 4, 2, 32)          # pair, low / high nibble, byte
        parts = [_half_bytes(d), _half_bytes(dm), _pack_sc_m(sc.to(torch.int32), mn.to(torch.int32))]
        if wtype == "q5_K":
            bits = torch.arange(8, device=x.device, dtype=torch.int32).reshape(1, 4, 2, 1)
            parts.append(((q >> 4) << bits).sum((1, 2)).to(torch.uint8))
        parts.append(((q[:, :, 0] & 15) | ((q[:, :, 1] & 15) << 4)).reshape(-1, 128).to(torch.uint8))
        raw = torch.cat(parts, 1)
    assert raw.shape[1] == size
    return raw.reshape(n, -1), val.reshape(n, -1)


def _chunks(rows, K):
    step = max(1, (1 << 26) // K)
    return [(r, min(step, rows - r)) for r in range(0, rows, step)]


def _weight(seed, name, wtype, K, rows):
    """The matrix's bytes, on the host."""
    return np.concatenate([_quantize(0.02 * _randn(seed, f"{name}:{r}", n, K), wtype)[0].cpu().numpy()
                           for r, n in _chunks(rows, K)])


def _times(seed, name, wtype, x, rows):
    """x W^T in 64 bits, for that matrix; x [T, K]."""
    K = x.shape[1]
    return torch.cat([x @ _quantize(0.02 * _randn(seed, f"{name}:{r}", n, K), wtype)[1].to(F64).T
                      for r, n in _chunks(rows, K)], 1)


def _norm_weight(seed, name, n):
    return 1 + 0.01 * _randn(seed, name, n)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.to(F64)


# ---------------------------------------------------------------------------------------------
# graphs over the C entry points

def _core():
    core = gl.libs()["core"]
    core.ggml_backend_graph_compute_async.restype = C.c_int
    core.ggml_backend_graph_compute_async.argtypes = [C.c_void_p, C.c_void_p]
    return core


_held = {}


def _backend():
    """One backend for the process, as a program keeps it."""
    if "backend" not in _held:
        _core()
        _held["backend"] = gl.hip_backend(0)
    return _held["backend"]


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


class _Graph:
    """A graph with its tensors; the device memory goes when the last view of it does."""

    def __init__(self):
        self.core, self.ctx, self.buf = _core(), None, None
        self.ctx = self.core.ggml_init(gl.ggml_init_params(8 << 20, None, True))
        self.gf = self.core.ggml_new_graph(self.ctx)
        self.data = []

    def __getattr__(self, name):
        fn = getattr(self.core, "ggml_" + name)
        return lambda *args: fn(self.ctx, *args)

    def tensor(self, ttype, ne, data=None):
        t = getattr(self.core, f"ggml_new_tensor_{len(ne)}d")(self.ctx, ttype, *ne)
        if data is not None:
            if isinstance(data, torch.Tensor):
                data = data.contiguous().cpu().numpy()
            self.data.append((t, np.ascontiguousarray(data)))
        return t

    def weight(self, seed, name, wtype, K, rows, experts=0):
        data = _weight(seed, name, wtype, K, rows * max(experts, 1))
        return self.tensor(TYPES[wtype], (K, rows, experts) if experts else (K, rows), data)

    def norm(self, x, seed, name, n, eps):
        return self.mul(self.rms_norm(x, eps), self.tensor(gl.F32, (n,), _norm_weight(seed, name, n)))

    def also(self, t):
        self.core.ggml_build_forward_expand(self.gf, t)

    def finish(self, out):
        self.core.ggml_set_output(out)
        self.also(out)
        self.buf = self.core.ggml_backend_alloc_ctx_tensors(self.ctx, _backend())
        if not self.buf:
            raise MemoryError("out of memory for a graph")
        for t, a in self.data:
            assert a.nbytes == self.core.ggml_nbytes(t)
            self.core.ggml_backend_tensor_set(t, _ptr(a), 0, a.nbytes)
        self.data = []

    def view(self, t, shape, half=False, offset=0):
        """The tensor's device memory as a torch tensor."""
        return torch.as_tensor(_Memory(self, t.contents.data + offset, shape, "<f2" if half else "<f4"), device=DEV)

    def __del__(self):
        if self.buf:
            self.core.ggml_backend_buffer_free(self.buf)
        if self.ctx:
            self.core.ggml_free(self.ctx)


class _Memory:
    def __init__(self, owner, data, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(data, False), version=3)


def _stream(seed, T, E):
    """T rows of a residual stream."""
    return _randn(seed, "x", T, E)


def _mask(past, T):
    q, k = torch.arange(T, device=DEV)[:, None], torch.arange(past + T, device=DEV)[None]
    return torch.where(k <= past + q, 0.0, -math.inf).float()


def _proj_graph(g, c, seed):
    x = g.tensor(gl.F32, (c["K"], c["T"]), _stream(seed, c["T"], c["K"]))
    y = g.mul_mat(g.weight(seed, "w", c["type"], c["K"], c["N"]), x)
    g.finish(y)
    return [g.view(y, (c["T"], c["N"]))]


def _proj_exact(c, seed):
    return [_times(seed, "w", c["type"], _stream(seed, c["T"], c["K"]).to(F64), c["N"])]


def _cache(c, seed, name, n_ctx):
    """A cache of n_ctx positions, the past ones filled."""
    h = HEADS[c["arch"]]
    kv = torch.zeros(n_ctx, h["head_kv"], h["hd"], device=DEV, dtype=torch.float16)
    kv[:c["past"]] = _randn(seed, name, c["past"], h["head_kv"], h["hd"]).to(torch.float16)
    return kv


def _attn_graph(g, c, seed):
    h, T, past, wt = HEADS[c["arch"]], c["T"], c["past"], c["type"]
    E, nh, nkv, hd, n_kv = h["embd"], h["head"], h["head_kv"], h["hd"], past + T
    x = g.tensor(gl.F32, (E, T), _stream(seed, T, E))
    pos = g.tensor(gl.I32, (T,), torch.arange(past, n_kv, dtype=torch.int32))
    mask = g.tensor(gl.F32, (n_kv, T), _mask(past, T))
    kc, vc = (g.tensor(gl.F16, (hd, nkv, n_kv), _cache(c, seed, n, n_kv)) for n in ("k", "v"))
    y = g.norm(x, seed, "norm", E, h["eps"])
    if h["fused"]:
        rows = (nh + 2 * nkv) * hd
        qkv = g.mul_mat(g.weight(seed, "qkv", wt, E, rows), y)
        q, k, v = (g.view_3d(qkv, hd, n, T, hd * 4, rows * 4, at * hd * 4)
                   for n, at in ((nh, 0), (nkv, nh), (nkv, nh + nkv)))
    else:
        q, k, v = (g.reshape_3d(g.mul_mat(g.weight(seed, w, wt, E, n * hd), y), hd, n, T)
                   for w, n in (("q", nh), ("k_w", nkv), ("v_w", nkv)))
    if h["qk_norm"]:
        q, k = g.norm(q, seed, "q_norm", hd, h["eps"]), g.norm(k, seed, "k_norm", hd, h["eps"])
    mode = gl.ROPE_NEOX if h["neox"] else gl.ROPE_NORMAL
    q, k = (g.rope_ext(t, pos, None, hd, mode, 131072, h["base"], 1.0, 0.0, 1.0, 0.0, 0.0) for t in (q, k))
    nb1, nb2 = hd * 2, hd * nkv * 2
    for new, cache in ((k, kc), (v, vc)):
        g.also(g.cpy(new, g.view_3d(cache, hd, nkv, T, nb1, nb2, past * nb2)))
    kf, vf = (g.view_3d(cache, hd, nkv, n_kv, nb1, nb2, 0) for cache in (kc, vc))
    kq = g.soft_max_ext(g.mul_mat(g.permute(kf, 0, 2, 1, 3), g.permute(q, 0, 2, 1, 3)), mask, 1 / math.sqrt(hd), 0.0)
    kqv = g.mul_mat(g.cont_3d(g.permute(vf, 1, 2, 0, 3), n_kv, hd, nkv), kq)
    out = g.mul_mat(g.weight(seed, "o", wt, nh * hd, E), g.cont_2d(g.permute(kqv, 0, 2, 1, 3), nh * hd, T))
    out = g.add(out, x)
    g.finish(out)
    return [g.view(out, (T, E))] + [g.view(cache, (T, nkv, hd), True, past * nb2) for cache in (kc, vc)]


def _rope64(x, past, base, neox):
    """RoPE of x [T, heads, hd] at positions past .. past + T - 1."""
    T, _, hd = x.shape
    freq = base ** (-2 * torch.arange(hd // 2, device=DEV, dtype=F64) / hd)
    a = (torch.arange(past, past + T, device=DEV, dtype=F64)[:, None] * freq)[:, None]
    cos, sin = a.cos(), a.sin()
    u, v = (x[..., :hd // 2], x[..., hd // 2:]) if neox else (x[..., 0::2], x[..., 1::2])
    r = (u * cos - v * sin, u * sin + v * cos)
    return torch.cat(r, -1) if neox else torch.stack(r, -1).reshape(x.shape)


def _attend64(q, k, v, past):
    """Causal attention of q [T, heads, hd] over k, v [past + T, kv heads, hd]."""
    T, nh, hd = q.shape
    group = nh // k.shape[1]
    mask = _mask(past, T).to(F64)
    return torch.cat([torch.softmax(q[:, i] @ k[:, i // group].T / math.sqrt(hd) + mask, 1) @ v[:, i // group]
                      for i in range(nh)], 1)


def _attn64(h, x, past, mm, nw, caches):
    """The attention half in 64 bits: mm(name, x, rows) is a product, nw(name, n) a norm weight and
    caches the filled K and V rows; the output and the new K and V rows."""
    T, (nh, nkv, hd) = x.shape[0], (h["head"], h["head_kv"], h["hd"])
    y = _rms(x, nw("norm", h["embd"]), h["eps"])
    if h["fused"]:
        q, k, v = mm("qkv", y, (nh + 2 * nkv) * hd).split((nh * hd, nkv * hd, nkv * hd), 1)
    else:
        q, k, v = mm("q", y, nh * hd), mm("k_w", y, nkv * hd), mm("v_w", y, nkv * hd)
    q, k, v = (t.reshape(T, -1, hd) for t in (q, k, v))
    if h["qk_norm"]:
        q, k = _rms(q, nw("q_norm", hd), h["eps"]), _rms(k, nw("k_norm", hd), h["eps"])
    q, k = _rope64(q, past, h["base"], h["neox"]), _rope64(k, past, h["base"], h["neox"])
    kf, vf = (torch.cat([old[:past].to(F64), new]) for old, new in zip(caches, (k, v)))
    return mm("o", _attend64(q, kf, vf, past), h["embd"]) + x, k, v


def _attn_exact(c, seed):
    h, T, past = HEADS[c["arch"]], c["T"], c["past"]
    return list(_attn64(h, _stream(seed, T, h["embd"]).to(F64), past,
                        lambda name, x, rows: _times(seed, name, c["type"], x, rows),
                        lambda name, n: _norm_weight(seed, name, n),
                        [_cache(c, seed, n, past) for n in ("k", "v")]))


def _ffn_graph(g, c, seed):
    E, F, T = c["embd"], c["ff"], c["T"]
    x = g.tensor(gl.F32, (E, T), _stream(seed, T, E))
    y = g.norm(x, seed, "norm", E, 1e-6)
    gate, up = (g.mul_mat(g.weight(seed, n, c["type"], E, F), y) for n in ("gate", "up"))
    act = g.mul(g.silu(gate), up)
    out = g.add(g.mul_mat(g.weight(seed, "down", c["type"], F, E), act), x)
    g.finish(out)
    return [g.view(out, (T, E))]


def _ffn64(x, F, mm, nw, eps):
    y = _rms(x, nw, eps)
    act = torch.nn.functional.silu(mm("gate", y, F)) * mm("up", y, F)
    return mm("down", act, x.shape[1]) + x


def _ffn_exact(c, seed):
    x = _stream(seed, c["T"], c["embd"]).to(F64)
    return [_ffn64(x, c["ff"], lambda name, v, rows: _times(seed, name, c["type"], v, rows),
                   _norm_weight(seed, "norm", c["embd"]), 1e-6)]


def _moe_graph(g, c, seed):
    E, F, T, X, k = c["embd"], c["ff"], c["T"], c["experts"], c["k"]
    x = g.tensor(gl.F32, (E, T), _stream(seed, T, E))
    y = g.norm(x, seed, "norm", E, 1e-6)
    probs = g.soft_max_ext(g.mul_mat(g.tensor(gl.F32, (E, X), 0.02 * _randn(seed, "router", X, E)), y), None, 1.0, 0.0)
    sel = g.top_k(probs, k)
    w = g.reshape_2d(g.get_rows(g.reshape_3d(probs, 1, X, T), sel), k, T)
    w = g.reshape_3d(g.div(w, g.sum_rows(w)), 1, k, T)
    y3 = g.reshape_3d(y, E, 1, T)
    gate, up = (g.mul_mat_id(g.weight(seed, n, c["type"], E, F, X), y3, sel) for n in ("gate", "up"))
    act = g.mul(g.silu(gate), up)
    parts = g.mul(g.mul_mat_id(g.weight(seed, "down", c["type"], F, E, X), act, sel), w)
    out = g.view_2d(parts, E, T, k * E * 4, 0)
    for i in range(1, k):
        out = g.add(out, g.view_2d(parts, E, T, k * E * 4, i * E * 4))
    out = g.add(out, x)
    g.finish(out)
    return [g.view(out, (T, E))]


def _moe_exact(c, seed):
    E, F, T, X, k = c["embd"], c["ff"], c["T"], c["experts"], c["k"]
    x = _stream(seed, T, E).to(F64)
    y = _rms(x, _norm_weight(seed, "norm", E), 1e-6)
    probs, sel = torch.softmax(y @ (0.02 * _randn(seed, "router", X, E)).to(F64).T, 1).topk(k, 1)
    w = probs / probs.sum(1, keepdim=True)
    mats = {n: torch.cat([_quantize(0.02 * _randn(seed, f"{n}:{r}", m, K), c["type"])[1]
                          for r, m in _chunks(rows * X, K)]).reshape(X, rows, K)
            for n, rows, K in (("gate", F, E), ("up", F, E), ("down", E, F))}
    out = x.clone()
    for e in range(X):
        t, slot = (sel == e).nonzero(as_tuple=True)
        if len(t):
            a = torch.nn.functional.silu(y[t] @ mats["gate"][e].to(F64).T) * (y[t] @ mats["up"][e].to(F64).T)
            out.index_add_(0, t, (a @ mats["down"][e].to(F64).T) * w[t, slot][:, None])
    return [out]


# ---------------------------------------------------------------------------------------------
# whole models

MODEL_SEED = 1   # the model file is the same for every prompt


def _model_mats(c):
    """(GGUF name, seeded name, row length, rows) of every matrix."""
    h, F, V = HEADS[c["arch"]], c["ff"], c["vocab"]
    E, q, kv = h["embd"], h["head"] * h["hd"], h["head_kv"] * h["hd"]
    mats = [("token_embd", "embd", E, V), ("output", "output", E, V)]
    for i in range(c["layers"]):
        mats += [(f"blk.{i}.{n}", f"{i}.{s}", K, rows) for n, s, K, rows in (
            ("attn_q", "q", E, q), ("attn_k", "k_w", E, kv), ("attn_v", "v_w", E, kv), ("attn_output", "o", q, E),
            ("ffn_gate", "gate", E, F), ("ffn_up", "up", E, F), ("ffn_down", "down", F, E))]
    return mats


def _model_norms(c):
    h = HEADS[c["arch"]]
    norms = [("output_norm", "output_norm", h["embd"])]
    for i in range(c["layers"]):
        norms += [(f"blk.{i}.attn_norm", f"{i}.norm", h["embd"]), (f"blk.{i}.ffn_norm", f"{i}.ffn_norm", h["embd"])]
        if h["qk_norm"]:
            norms += [(f"blk.{i}.attn_{n}_norm", f"{i}.{n}_norm", h["hd"]) for n in ("q", "k")]
    return norms


def _model_file(c):
    """The model of this case as a GGUF file, written once for the process."""
    key = tuple(sorted((k, v) for k, v in c.items() if k not in ("name", "past", "T")))
    if key in _held:
        return _held[key]
    if "dir" not in _held:
        _held["dir"] = tempfile.TemporaryDirectory()
    core, h = _core(), HEADS[c["arch"]]
    path = os.path.join(_held["dir"].name, f"{len(_held)}.gguf")
    ctx = core.ggml_init(gl.ggml_init_params(8 << 20, None, True))
    f = core.gguf_init_empty()
    arch = c["arch"]
    core.gguf_set_val_str(f, b"general.architecture", arch.encode())
    for key_, v in (("embedding_length", h["embd"]), ("block_count", c["layers"]), ("context_length", 32768),
                    ("feed_forward_length", c["ff"]), ("attention.head_count", h["head"]),
                    ("attention.head_count_kv", h["head_kv"]), ("attention.key_length", h["hd"]),
                    ("rope.dimension_count", h["hd"])):
        core.gguf_set_val_u32(f, f"{arch}.{key_}".encode(), v)
    core.gguf_set_val_f32(f, f"{arch}.attention.layer_norm_rms_epsilon".encode(), h["eps"])
    core.gguf_set_val_f32(f, f"{arch}.rope.freq_base".encode(), h["base"])
    held = [(n, TYPES[c["type"]], (K, rows), _weight(MODEL_SEED, s, c["type"], K, rows)) for n, s, K, rows in _model_mats(c)]
    held += [(n, gl.F32, (k,), _norm_weight(MODEL_SEED, s, k).cpu().numpy()) for n, s, k in _model_norms(c)]
    for name, ttype, ne, data in held:
        t = getattr(core, f"ggml_new_tensor_{len(ne)}d")(ctx, ttype, *ne)
        core.ggml_set_name(t, f"{name}.weight".encode())
        t.contents.data = data.ctypes.data
        core.gguf_add_tensor(f, t)
    ok = core.gguf_write_to_file(f, path.encode(), False)
    core.gguf_free(f)
    core.ggml_free(ctx)
    if not ok:
        raise OSError("cannot write " + path)
    _held[key] = path
    return path


def _prompt(c, seed):
    return torch.randint(0, c["vocab"], (c["past"] + c["T"],), generator=_gen(seed, "prompt"), device=DEV)


def _model_exact(c, seed):
    h = HEADS[c["arch"]]
    tokens, wt = _prompt(c, seed), c["type"]
    x = torch.zeros(len(tokens), h["embd"], device=DEV, dtype=F64)
    for r, n in _chunks(c["vocab"], h["embd"]):
        rows = _quantize(0.02 * _randn(MODEL_SEED, f"embd:{r}", n, h["embd"]), wt)[1]
        here = (tokens >= r) & (tokens < r + n)
        x[here] = rows[tokens[here] - r].to(F64)
    for i in range(c["layers"]):
        mm = lambda name, v, rows: _times(MODEL_SEED, f"{i}.{name}", wt, v, rows)  # noqa: E731
        nw = lambda name, n: _norm_weight(MODEL_SEED, f"{i}.{name}", n)  # noqa: E731
        empty = torch.zeros(0, h["head_kv"], h["hd"], device=DEV)
        x = _attn64(h, x, 0, mm, nw, (empty, empty))[0]
        x = _ffn64(x, c["ff"], mm, nw("ffn_norm", h["embd"]), h["eps"])
    y = _rms(x[-1:], _norm_weight(MODEL_SEED, "output_norm", h["embd"]), h["eps"])
    return [_times(MODEL_SEED, "output", wt, y, c["vocab"])[0]]


# ---------------------------------------------------------------------------------------------
# what the measurement calls

GRAPHS = {"proj": _proj_graph, "attn": _attn_graph, "ffn": _ffn_graph, "moe": _moe_graph}
EXACT = {"proj": _proj_exact, "attn": _attn_exact, "ffn": _ffn_exact, "moe": _moe_exact, "model": _model_exact}


class _Session:
    """A session whose cache holds the prompt's first `past` tokens, and its next T tokens."""

    def __init__(self, c, seed):
        prompt = _prompt(c, seed).to(torch.int32).cpu().numpy()
        self.past, self.tokens = c["past"], prompt[c["past"]:]
        self.session = gl.Session(_model_file(c), "hip", n_ctx=len(prompt))
        if self.past:
            self.session.forward(0, prompt[:self.past])

    def __del__(self):
        self.session.close()


def prepare(case, seed):
    if case["kind"] == "model":
        return _Session(case, seed)
    g = _Graph()
    g.outputs = GRAPHS[case["kind"]](g, case, seed)
    state = (g, _backend(), g.outputs)
    g.outputs = None
    return state


def run(state):
    if isinstance(state, _Session):
        return [state.session.forward(state.past, state.tokens)]
    g, backend, outputs = state
    if g.core.ggml_backend_graph_compute_async(backend, g.gf) != 0:
        raise RuntimeError("graph compute failed")
    return outputs


def exact(case, seed):
    return EXACT[case["kind"]](case, seed)


def _mat_work(wtype, K, rows, T):
    qk, size = BLOCK[wtype]
    return rows * (K // qk) * size, 2 * K * rows * T


def _attn_work(h, wtype, past, T):
    E, q, kv = h["embd"], h["head"] * h["hd"], h["head_kv"] * h["hd"]
    b, f = (sum(v) for v in zip(_mat_work(wtype, E, q + 2 * kv, T), _mat_work(wtype, q, E, T)))
    pairs = T * past + T * (T + 1) // 2
    return b + 2 * (past + T) * kv * 2 + 8 * T * E, f + 4 * pairs * q


def _ffn_work(wtype, E, F, T):
    b, f = (sum(v) for v in zip(_mat_work(wtype, E, 2 * F, T), _mat_work(wtype, F, E, T)))
    return b + 8 * T * E, f


def work(case):
    """Weights, cache, inputs and outputs once each; the products' operations."""
    c = case
    wt, T, kind = c["type"], c["T"], c["kind"]
    if kind == "proj":
        b, f = _mat_work(wt, c["K"], c["N"], T)
        b += 4 * T * (c["K"] + c["N"])
    elif kind == "attn":
        b, f = _attn_work(HEADS[c["arch"]], wt, c["past"], T)
    elif kind == "ffn":
        b, f = _ffn_work(wt, c["embd"], c["ff"], T)
    elif kind == "moe":
        # the experts that some token is routed to, with even routing
        used = c["experts"] * (1 - (1 - c["k"] / c["experts"]) ** T)
        b, f = _ffn_work(wt, c["embd"], c["ff"], T)
        b = (b - 8 * T * c["embd"]) * used + 4 * c["embd"] * (c["experts"] + 2 * T)
        f = f * c["k"] + 2 * c["embd"] * c["experts"] * T
    else:
        h = HEADS[c["arch"]]
        parts = [_attn_work(h, wt, c["past"], T), _ffn_work(wt, h["embd"], c["ff"], T)]
        b, f = (sum(v) * c["layers"] for v in zip(*parts))
        hb, hf = _mat_work(wt, h["embd"], c["vocab"], T)
        b, f = b + hb + 4 * c["vocab"], f + hf
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    """About four times what a last-bit change is seen to travel to the outputs. A product's sums in
    another order: 2e-7. A block's input off by one unit in the last place moves some values across a
    rounding step of the next 8-bit quantization: up to 4.3e-4. A model's norm weights so: 4e-2."""
    if case["kind"] == "proj":
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] == "model":
        return {"rel": 3e-2, "max": 0.9}
    return {"rel": 1.5e-3, "max": 6e-2}
