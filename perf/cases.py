"""Timed cases of the attention path and the layers around it, each one pass of a model layer.

A case is one call that a model's forward makes per layer: the fused head norms + RoPE + K/V store
+ attention on the packed qkv_proj output (``Attention.forward_packed_qkv``), over the step that the
engine set on the context, or ``o_proj`` on the attention output (``Linear.forward``).  Head shapes
are those of the model families the library serves:

=========  ==================  ==========================================================
``style``  q heads/KV heads/d  head norms, as the model layers apply them
=========  ==================  ==========================================================
qwen3      16/8/128, 32/8/128, q and k RMSNorm
           40/8/128
llama      32/8/64             none
gemma3     4/1/256             q and k RMSNorm with (1 + w), scale 1/16
gemma4     8/1/512             q and k RMSNorm, weightless v RMSNorm, scale 1
=========  ==================  ==========================================================

Sequences are written ``cached+new`` (tokens already in the pages, tokens of this step); decode rows
are given by their number and the range of their context lengths.  ``layout`` seeds the lengths;
the inputs, the pages' contents and their order in the arena come from the seed of ``prepare``.
"""

import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "nano-vllm-java_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from nanollvm_amd import Attention, Context, KvCacheArena, Linear, RMSNorm, RotaryEmbedding  # noqa: E402
from nanollvm_amd import workloads as W  # noqa: E402

EPS = 1e-6
MAX_POS = 40960

# q heads, KV heads, head dim, RoPE theta, and the families' head norms.
SHAPES = {
    "qwen3-0.6b": dict(hq=16, hkv=8, d=128, theta=1e6, style="qwen3"),
    "qwen3-4b": dict(hq=32, hkv=8, d=128, theta=1e6, style="qwen3"),
    "qwen3-14b": dict(hq=40, hkv=8, d=128, theta=1e6, style="qwen3"),
    "llama": dict(hq=32, hkv=8, d=64, theta=5e5, style="llama"),
    "gemma3": dict(hq=4, hkv=1, d=256, theta=1e6, style="gemma3"),
    "gemma4": dict(hq=8, hkv=1, d=512, theta=1e6, style="gemma4"),
}


def _attn(name, shape, *, seqs="", rows=0, lo=0, hi=0, window=0, block=256, layout=0):
    """One attention layer pass: prefill sequences (``seqs``) and / or ``rows`` decode rows with
    contexts in [lo, hi] (uniform within a factor of four, log-uniform beyond)."""
    case = dict(kind="attention", shape=shape, seqs=seqs, rows=rows, lo=lo, hi=hi, window=window,
                block=block, layout=layout)
    if name:
        case["name"] = name
    return case


def _linear(name, rows, inf, outf, bias=False):
    case = dict(kind="linear", rows=rows, inf=inf, outf=outf, bias=bias)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # A chat server with few users: eight rows, short contexts, launches and latency count.
        _attn("decode_8_rows", "qwen3-0.6b", rows=8, lo=256, hi=1024),
        # A full decode batch at mixed contexts up to 32K: 15 GB of K/V per layer pass.
        _attn("decode_256_rows", "qwen3-0.6b", rows=256, lo=128, hi=32768),
        # Multi-query decode of a small Gemma, full-attention layer.
        _attn("decode_gemma3_global", "gemma3", rows=32, lo=512, hi=8192),
        # Five query heads per KV head, a medium batch with long contexts.
        _attn("decode_48_rows_gqa5", "qwen3-14b", rows=48, lo=256, hi=32768),
        # Fresh short prompts of odd lengths, nothing cached (attention over the step's own rows).
        _attn("prefill_short_prompts", "llama", seqs="0+17,0+201,0+64,0+333,0+5,0+127,0+96"),
        # Four prompts, the last continuing after a prefix found in the cache.
        _attn("prefill_varlen_prefix", "qwen3-0.6b", seqs="0+512,0+1024,0+1536,1024+1024"),
        # A late chunk of one long prompt.
        _attn("prefill_long_chunk", "qwen3-4b", seqs="12289+2048"),
        # Sliding-window layer of a Gemma, fresh prompts.
        _attn("prefill_gemma3_local", "gemma3", seqs="0+512,0+1024,0+1536,0+2048", window=512),
        # Full-attention layer with wide heads.
        _attn("prefill_gemma4_global", "gemma4", seqs="0+512,0+1024,0+1536,0+2048"),
        # Chunked prefill: four chunks share the step with 64 decode rows.
        _attn("mixed_chunks_rows", "qwen3-4b", seqs="2601+512,1893+512,3391+512,251+512", rows=64,
              lo=4096, hi=16384),
        # o_proj of a decode batch and of a prefill step.
        _linear("o_proj_200_rows", 200, 2048, 1024),
        _linear("o_proj_4096_rows", 4096, 2048, 1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: any head shape, batch, lengths, page size and window; no larger
    than the largest listed one."""
    while True:
        case = _draw(rng)
        w = work(case)
        if w["bytes"] <= 12e9 and w["flops"] <= 300e9:
            return case


def _draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed", "linear"])
    if kind == "linear":
        inf, outf = rng.choice([(2048, 1024), (4096, 2560), (2048, 2048), (1024, 640),
                                (5120, 5120), (4096, 1152), (1028, 1000)])
        return _linear(None, _log(rng, 1, 4500), inf, outf, rng.random() < 0.3)
    shape = rng.choice(sorted(SHAPES))
    window = rng.choice([0, 0, 512, 1024]) if shape == "gemma3" else 0
    block = rng.choice([256, 256, 64, 16])
    layout = rng.randrange(1 << 20)
    if kind == "decode":
        lo = _log(rng, 16, 4096)
        return _attn(None, shape, rows=_log(rng, 1, 256), lo=lo, hi=min(32768, lo * _log(rng, 2, 64)),
                     window=window, block=block, layout=layout)
    fresh = rng.random() < 0.4
    total, seqs = _log(rng, 40, 6000), []
    while total > 0 and len(seqs) < 12:
        n = min(total, _log(rng, 2, 3000))
        cached = 0 if fresh or rng.random() < 0.5 else _log(rng, 1, 8000)
        seqs.append(f"{cached}+{n}")
        total -= n
    if kind == "prefill":
        return _attn(None, shape, seqs=",".join(seqs), window=window, block=block, layout=layout)
    lo = _log(rng, 64, 4096)
    return _attn(None, shape, seqs=",".join(seqs), rows=_log(rng, 2, 96), lo=lo,
                 hi=min(32768, lo * _log(rng, 2, 16)), window=window, block=block, layout=layout)


@functools.lru_cache(maxsize=64)
def _lengths(seqs, rows, lo, hi, layout):
    """(cached, new) of every sequence of the step, the decode rows last."""
    got = [tuple(int(x) for x in s.split("+")) for s in seqs.split(",") if s]
    rng = np.random.default_rng(layout)
    if rows:
        lens = (W.uniform_lengths if hi <= 4 * lo else W.loguniform_lengths)(rng, rows, lo, hi)
        got += [(c - 1, 1) for c in lens]
    return tuple(got)


def _seqs(case):
    return list(_lengths(case["seqs"], case["rows"], case["lo"], case["hi"], case["layout"]))


def _dense(case):
    """Nothing of the step's sequences is cached: the engine attaches no block tables, and
    attention runs over the step's own rows."""
    return bool(case["seqs"]) and all(c == 0 for c, _ in _seqs(case))


def _workload(case, seed):
    s = SHAPES[case["shape"]]
    seqs = _seqs(case)
    style = s["style"]
    scale = 1.0 if style == "gemma4" else s["d"] ** -0.5
    return W.build(case["shape"], seqs, is_prefill=bool(case["seqs"]), hq=s["hq"], hkv=s["hkv"],
                   d=s["d"], scale=scale, window=case["window"],
                   rng=np.random.default_rng(seed), block_size=case["block"],
                   pool_cap=W.POOL_CAP * (256 // case["block"]), rope_theta=s["theta"],
                   max_pos=MAX_POS)


@functools.lru_cache(maxsize=8)
def _table(d, theta):
    """[MAX_POS, d] cos | sin table of the model, as its loader builds it."""
    inv = (1.0 / theta ** (np.arange(0, d, 2) / d)).astype(np.float32)
    ang = (np.arange(MAX_POS, dtype=np.float32)[:, None] * inv[None, :]).astype(np.float64)
    return np.concatenate([np.cos(ang), np.sin(ang)], axis=1).astype(np.float32)


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 16 + salt)
    return g


def _fill(flat, seed, salt):
    g = _gen(seed, salt)
    for s in range(0, flat.numel(), 1 << 28):
        flat[s:s + (1 << 28)].normal_(generator=g)


def _weights(case, seed):
    """The model's head-norm weights: (q, k, adds one) or None."""
    s = SHAPES[case["shape"]]
    if s["style"] == "llama":
        return None
    g = _gen(seed, 1)
    noise = 0.1 * torch.randn(2, s["d"], device="cuda", generator=g)
    if s["style"] == "gemma4":  # scale 1: the learned gains keep the scores small
        return 0.3 * (1.0 + noise[0]), 0.3 * (1.0 + noise[1]), False
    if s["style"] == "gemma3":
        return 0.3 + noise[0], 0.3 + noise[1], True
    return 1.4 + noise[0], 1.2 + noise[1], False


def _qkv(case, tokens, seed):
    s = SHAPES[case["shape"]]
    return torch.randn(tokens, (s["hq"] + 2 * s["hkv"]) * s["d"], device="cuda",
                       generator=_gen(seed, 2))


class _Engine:
    """The objects an engine keeps: context, arena, RoPE table.  Closed with the last user of the
    pages (a state, or a tensor over the pages)."""

    def __init__(self, case, wl):
        self.ctx = Context(0)
        self.arena = KvCacheArena(self.ctx, 1, wl.num_blocks, wl.block_size, wl.hkv, wl.d)
        self.rope = RotaryEmbedding(self.ctx, wl.d, wl.d, MAX_POS, wl.rope_theta,
                                    cos_sin=_table(wl.d, wl.rope_theta))

    def pages(self):
        k, v, nbytes = self.arena.device_ptrs(0)
        return [torch.as_tensor(_Memory(p, nbytes // 4, self), device="cuda")
                .view(self.arena.num_blocks, -1) for p in (k, v)]

    def __del__(self):
        for name in ("rope", "arena", "ctx"):
            x = getattr(self, name, None)
            if x is not None:
                x.close()


class _Memory:
    """Device memory of the arena as torch.as_tensor takes it; keeps its owner alive."""

    def __init__(self, ptr, count, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f4",
                                         "data": (ptr, False), "version": 2, "strides": None}


class _AttentionState:
    def __init__(self, case, seed):
        wl = _workload(case, seed)
        self.engine = _Engine(case, wl)
        self.ctx = self.engine.ctx
        self.pages = self.engine.pages()
        for salt, p in zip((3, 4), self.pages):
            _fill(p.view(-1), seed, salt)
        w = _weights(case, seed)
        self.q_norm = None if w is None else RMSNorm(w[0], EPS, w[2])
        self.k_norm = None if w is None else RMSNorm(w[1], EPS, w[2])
        self.v_norm = RMSNorm.weightless(EPS) if SHAPES[case["shape"]]["style"] == "gemma4" else None
        self.attn = Attention(wl.hq, wl.d, wl.scale, wl.hkv, wl.window, 0)
        self.qkv = _qkv(case, wl.tokens, seed)
        meta = wl.meta
        if _dense(case):
            meta.block_tables = None
        self.ctx.set(**meta.context_args())
        self.ctx.bind_kv_cache(self.engine.arena)

    def run(self):
        out = self.attn.forward_packed_qkv(self.engine.rope, None, self.qkv, self.ctx,
                                           q_norm=self.q_norm, k_norm=self.k_norm,
                                           v_norm=self.v_norm)
        return {"out": out, "k": self.pages[0], "v": self.pages[1]}


def _linear_inputs(case, seed):
    x = torch.randn(case["rows"], case["inf"], device="cuda", generator=_gen(seed, 5))
    w = torch.randn(case["outf"], case["inf"], device="cuda", generator=_gen(seed, 6))
    w *= case["inf"] ** -0.5
    b = torch.randn(case["outf"], device="cuda", generator=_gen(seed, 7)) if case["bias"] else None
    return x, w, b


class _LinearState:
    def __init__(self, case, seed):
        self.ctx = Context(0)
        self.x, w, b = _linear_inputs(case, seed)
        self.layer = Linear(w, b)

    def run(self):
        return {"y": self.layer.forward(self.x, self.ctx)}

    def __del__(self):
        if getattr(self, "ctx", None) is not None:
            self.ctx.close()


def prepare(case, seed):
    return (_LinearState if case["kind"] == "linear" else _AttentionState)(case, seed)


def run(state):
    return state.run()


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["rows"], case["inf"], case["outf"]
        return {"bytes": 4.0 * (m * k + n * k + m * n), "flops": 2.0 * m * n * k}
    s = SHAPES[case["shape"]]
    hq, hkv, d, win = s["hq"], s["hkv"], s["d"], case["window"]
    tokens = pairs = keys = 0
    for c, n in _seqs(case):
        tokens += n
        vis = np.arange(c + 1, c + n + 1, dtype=np.int64)
        pairs += int(np.minimum(vis, win).sum() if win else vis.sum())
        if not _dense(case):  # cached keys some query of the step sees
            keys += c - max(0, c + 1 - win) if win else c
    # qkv read, the attention output and the new k / v rows written, the cached rows read.
    moved = tokens * (hq + 2 * hkv) * d + tokens * hq * d + 2 * (tokens + keys) * hkv * d
    return {"bytes": 4.0 * moved, "flops": 4.0 * d * hq * pairs}


def tolerance(case):
    # 32-bit sums throughout: against 64 bits the outputs are off by 2e-7 (decode) to 1.7e-6 (a
    # long prefill chunk's sums over 14K keys), and another summation order by as much again.
    return {"rel": 6e-6, "max": 2e-4}


def _rope(x, positions, table):
    d = x.shape[-1]
    cs = table[positions][:, None, :]
    c, s = cs[..., :d // 2], cs[..., d // 2:]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _rms(x, w=None, one_plus=False):
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + float(np.float32(EPS)))
    return y if w is None else y * (w.double() + 1.0 if one_plus else w.double())


def exact(case, seed):
    if case["kind"] == "linear":
        x, w, b = _linear_inputs(case, seed)
        y = x.double() @ w.double().T.contiguous()
        return {"y": y if b is None else y + b.double()}
    wl = _workload(case, seed)
    hq, hkv, d = wl.hq, wl.hkv, wl.d
    T, bs, rep = wl.tokens, wl.block_size, wl.hq // wl.hkv
    x = _qkv(case, T, seed).double().view(T, hq + 2 * hkv, d)
    q, k, v = x[:, :hq], x[:, hq:hq + hkv], x[:, hq + hkv:]
    w = _weights(case, seed)
    if w is not None:
        q, k = _rms(q, w[0], w[2]), _rms(k, w[1], w[2])
    if SHAPES[case["shape"]]["style"] == "gemma4":
        v = _rms(v)
    table = torch.from_numpy(_table(d, wl.rope_theta)).cuda().double()
    pos = torch.from_numpy(wl.meta.positions.astype(np.int64)).cuda()
    q, k = _rope(q, pos, table), _rope(k, pos, table)
    pages = []
    slots = torch.from_numpy(wl.meta.slot_mapping.astype(np.int64)).cuda()
    for salt, new in ((3, k), (4, v)):
        p = torch.empty(wl.num_blocks * bs * hkv * d, device="cuda")
        _fill(p, seed, salt)
        p = p.double().view(wl.num_blocks * bs, hkv, d)
        p[slots] = new
        pages.append(p)
    out = torch.empty(T, hq, d, dtype=torch.float64, device="cuda")
    scale = float(np.float32(wl.scale))
    at = 0
    for b, (c, n) in enumerate(wl.seqs):
        first = max(0, c + 1 - wl.window) if wl.window else 0  # the first key any query sees
        t = np.arange(first, c + n)
        rows = torch.from_numpy(np.asarray(wl.tables[b], np.int64)[t // bs] * bs + t % bs).cuda()
        key = torch.from_numpy(t).cuda()
        kk = pages[0][rows].permute(1, 2, 0).contiguous()  # [hkv, d, keys]
        vv = pages[1][rows].permute(1, 0, 2).contiguous()  # [hkv, keys, d]
        for t0 in range(0, n, 1024):
            t1 = min(n, t0 + 1024)
            aq = torch.arange(c + t0, c + t1, device="cuda")
            seen = key[None, :] <= aq[:, None]
            if wl.window:
                seen &= key[None, :] > aq[:, None] - wl.window
            for h in range(hkv):
                qh = q[at + t0:at + t1, h * rep:(h + 1) * rep].transpose(0, 1).reshape(-1, d)
                sc = (qh.contiguous() @ kk[h]).view(rep, t1 - t0, -1) * scale
                sc.masked_fill_(~seen[None], -math.inf)
                o = torch.softmax(sc, dim=-1).view(rep * (t1 - t0), -1) @ vv[h]
                out[at + t0:at + t1, h * rep:(h + 1) * rep] = \
                    o.view(rep, t1 - t0, d).transpose(0, 1)
        at += n
    return {"out": out, "k": pages[0].view(wl.num_blocks, -1), "v": pages[1].view(wl.num_blocks, -1)}
