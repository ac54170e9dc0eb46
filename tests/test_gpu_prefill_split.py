"""Prefill on split fp16 operands at magnitudes where the split can go wrong.

The kernel scales q per query and K / V per 32-key tile by powers of two and takes queries whose
results are small beside their tiles again on fp32 instructions.  Each case is compared row by row
(rel-L2 of every query row of every head), so that a small row beside a large one counts by itself:
with float64 where the inputs are finite, with the oracle where they are not (non-finite results
must be the oracle's).  Bar: 1e-5, the attention bar: up to 2100 fp32 products per output give
sqrt(2100) * 2^-24 = 2.7e-6 of their size, a few times that where they cancel, and a score of size
s < 10 moves its weight by s times its own error.  (The fp32 oracle itself is 2.0e-5 off on the
long rows of unlike size.)"""

import numpy as np
import pytest
import torch

from cases import Case
from gpu_checks import dev, load_arena, say
from nanollvm_amd import Attention, Context, KvCacheArena
from nanollvm_amd import workloads as W

pytestmark = pytest.mark.gpu

# The last sequence gives the step work enough for the split kernel (steps of short sequences run
# on the fp32 one; every case checks which one ran).  A window leaves few keys per query, so it
# takes more queries.
SEQS = [(16, 70), (5, 33), (0, 2), (40, 190), (0, 31)]
DENSE_SEQS = [(0, 70), (0, 33), (0, 2), (0, 190), (0, 31)]
LONG, LONG_WINDOW = [(0, 2100)], [(0, 9000)]
HEADS = [(64, 1), (64, 4), (128, 1), (128, 2), (256, 1), (256, 4), (512, 1), (512, 2)]


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def build(d, rep, layout, window=0, scale=None, seed=0):
    rng = np.random.default_rng(seed + d + rep)
    paged = layout != "dense"
    wl = W.build(f"split d{d} rep{rep} {layout} w{window}",
                 (SEQS if paged else DENSE_SEQS) + (LONG_WINDOW if window else LONG),
                 is_prefill=True, hq=2 * rep, hkv=2, d=d,
                 scale=float(np.float32(scale if scale is not None else d ** -0.5)),
                 window=window, rng=rng, paged=paged,
                 block_size=int(layout[5:]) if paged else 256, pool_cap=20000)
    return Case(wl, seed=seed)


def exact(case, kc, vc):
    """The step's attention in float64."""
    wl, m = case.wl, case.wl.meta
    rep = wl.hq // wl.hkv
    out = np.zeros(case.q.shape)
    for b, (c, n) in enumerate(wl.seqs):
        q0 = int(m.cu_seqlens_q[b])
        if wl.tables is None:
            k, v = case.k[q0:q0 + n], case.v[q0:q0 + n]
        else:
            t = np.arange(c + n)
            rows = np.asarray(wl.tables[b], np.int64)[t // wl.block_size] * wl.block_size
            rows += t % wl.block_size
            k, v = (x.reshape(-1, wl.hkv, wl.d)[rows] for x in (kc, vc))
        k, v, q = (torch.from_numpy(x).cuda().double() for x in (k, v, case.q[q0:q0 + n]))
        at = torch.arange(c, c + n, device="cuda")[:, None]
        key = torch.arange(c + n, device="cuda")[None, :]
        seen = (key <= at) & ((key > at - wl.window) if wl.window else True)
        for h in range(wl.hq):
            kt = k[:, h // rep].T.contiguous()
            s = (q[:, h].contiguous() @ kt * wl.scale).masked_fill(~seen, -np.inf)
            p = torch.softmax(s, dim=-1)
            out[q0:q0 + n, h] = (p @ v[:, h // rep].contiguous()).cpu().numpy()
    return out


def check(ctx, case, name):
    wl = case.wl
    say(name)
    arena = load_arena(ctx, case)
    try:
        ctx.set(**wl.meta.context_args())
        ctx.bind_kv_cache(arena)
        with np.errstate(all="ignore"):
            want, kc, vc = case.oracle(threads=8)
        ctx.reset_stats()
        ctx.set_timing(True)
        out = Attention(wl.hq, wl.d, wl.scale, wl.hkv, wl.window, 0).forward(
            dev(case.q), dev(case.k), dev(case.v), ctx)
        ctx.sync()
        got = out.cpu().numpy().astype(np.float64)
        launches, _ = ctx.kernel_stats("prefill_split")
        assert launches == 1, "the split kernel did not run"
    finally:
        ctx.set_timing(False)
        ctx.clear()
        arena.close()
    finite = all(np.isfinite(x).all() for x in (case.q, case.k, case.v))
    want = exact(case, kc, vc) if finite else want.astype(np.float64)
    odd = ~np.isfinite(want)
    assert np.array_equal(got[odd], want[odd], equal_nan=True), "non-finite results differ"
    assert np.all(np.isfinite(got[~odd])), "non-finite results where the oracle's are finite"
    got[odd] = want[odd] = 0.0
    err = np.linalg.norm(got - want, axis=-1)
    size = np.linalg.norm(want, axis=-1)
    rel = float(np.max(err / np.where(size > 0, size, 1.0)))
    say(f"{name}: worst row rel_l2={rel:.3e}")
    assert rel <= 1e-5, rel


@pytest.mark.parametrize("layout", ["paged8", "paged16", "paged24", "paged4", "dense", "paged32",
                                    "paged64", "paged256"])
@pytest.mark.parametrize("window", [0, 37])
@pytest.mark.parametrize("d,rep", HEADS)
def test_page_sizes_and_window_starts(ctx, d, rep, window, layout):
    """Full tiles inside one page and, over smaller pages of 8 tokens and more, aligned ones are read
    by whole runs; other sizes, unaligned window starts and the last tile row by row."""
    check(ctx, build(d, rep, layout, window, seed=1), f"pages d{d} rep{rep} w{window} {layout}")


@pytest.mark.parametrize("window", [0, 37])
@pytest.mark.parametrize("d,rep", [(64, 2), (64, 8), (128, 4), (128, 8), (256, 2), (256, 8), (512, 4),
                                   (512, 8)])
def test_other_head_ratios(ctx, d, rep, window):
    check(ctx, build(d, rep, "paged16", window, seed=8), f"heads d{d} rep{rep} w{window}")


@pytest.mark.parametrize("layout", ["paged16", "dense"])
@pytest.mark.parametrize("d,rep", HEADS)
def test_rows_of_unlike_size(ctx, d, rep, layout):
    """K and V rows over 2^-6 .. 2^6 (within one scale's span), q rows over 2^-30 .. 2^0, and
    whole sequences of V 2^+-50 apart (each its own tiles)."""
    case = build(d, rep, layout, seed=2)
    rng = np.random.default_rng(3)
    T = case.wl.tokens
    case.q *= np.exp2(rng.integers(-30, 1, (T, 1, 1))).astype(np.float32)
    case.k *= np.exp2(rng.integers(-6, 2, (T, 1, 1))).astype(np.float32)
    case.v *= np.exp2(rng.integers(-6, 7, (T, 1, 1))).astype(np.float32)
    cu = case.wl.meta.cu_seqlens_q
    for b in range(len(cu) - 1):
        case.v[cu[b]:cu[b + 1]] *= np.float32(2.0 ** (50 if b % 2 else -50))
        if case.paged:  # the sequence's cached rows with it
            bs = case.wl.block_size
            t = np.arange(case.wl.seqs[b][0])
            rows = np.asarray(case.wl.tables[b], np.int64)[t // bs] * bs + t % bs
            flat = case.v_cache.reshape(-1, case.wl.hkv, d)
            flat[rows] *= np.float32(2.0 ** (50 if b % 2 else -50))
    check(ctx, case, f"unlike rows d{d} rep{rep} {layout}")


@pytest.mark.parametrize("layout", ["paged16", "dense"])
@pytest.mark.parametrize("d,rep", HEADS)
def test_rows_beyond_one_scale(ctx, d, rep, layout):
    """One K row of 2^40 that every query weighs at 0, one V row of 2^60 late in the same tile
    (queries before it must keep the bits of their own rows) and a sequence whose first V row,
    in the dense layout all that its first query sees, is 2^-40 beside its tile's others."""
    case = build(d, rep, layout, seed=4)
    first = int(case.wl.meta.cu_seqlens_q[3])
    case.q[:, :, 0] = np.abs(case.q[:, :, 0]) + 0.5
    case.k[first + 9] = 0.0
    case.k[first + 9, :, 0] = -2.0 ** 40
    case.v[first + 20] *= np.float32(2.0 ** 60)
    case.v[0] *= np.float32(2.0 ** -40)
    check(ctx, case, f"beyond one scale d{d} rep{rep} {layout}")


@pytest.mark.parametrize("layout", ["paged16", "dense"])
@pytest.mark.parametrize("value,window", [(np.inf, 0), (np.nan, 0), (-np.inf, 37)])
@pytest.mark.parametrize("d,rep", HEADS)
def test_infinities(ctx, d, rep, value, window, layout):
    """An infinite (or NaN) V element reaches the queries that see it and no other; a key whose score
    is -inf has weight 0."""
    case = build(d, rep, layout, window, seed=5)
    first = int(case.wl.meta.cu_seqlens_q[3])
    case.q[:, :, 0] = np.abs(case.q[:, :, 0]) + 0.5
    case.v[first + 100, :, 3] = value
    case.k[first + 7] = 0.0
    case.k[first + 7, :, 0] = -np.inf
    check(ctx, case, f"infinities d{d} rep{rep} {value} w{window} {layout}")


@pytest.mark.parametrize("d,rep", [(128, 2), (256, 1), (512, 1)])
def test_more_segments_than_bits(ctx, d, rep):
    """Hundreds of short sequences, over 64 to a workgroup, and in some of them an infinity: a wave
    remembers the segments it takes again in 64 bits."""
    rng = np.random.default_rng(d)
    seqs = [(0, int(n)) for n in rng.integers(2, 7, 1500)] + LONG
    wl = W.build(f"many segments d{d}", seqs, is_prefill=True, hq=16 * rep, hkv=16, d=d,
                 scale=float(np.float32(d ** -0.5)), rng=rng, block_size=16, pool_cap=20000)
    case = Case(wl, seed=9)
    for b in (3, 700, 1400):
        case.v[int(wl.meta.cu_seqlens_q[b]), :, 5] = np.inf
    check(ctx, case, wl.name)


@pytest.mark.parametrize("d,rep", HEADS)
def test_zeros_and_negative_scale(ctx, d, rep):
    case = build(d, rep, "paged16", scale=-(d ** -0.5), seed=6)
    check(ctx, case, f"negative scale d{d} rep{rep}")
    case = build(d, rep, "dense", seed=7)
    case.k[:40] = 0.0
    case.v[20:90] = 0.0
    case.q[60:300] = 0.0
    check(ctx, case, f"zeros d{d} rep{rep}")


@pytest.mark.parametrize("d,hq,hkv,short,long", [(64, 32, 8, 70, 700), (128, 16, 8, 60, 600),
                                                 (512, 8, 1, 30, 600), (256, 4, 1, None, 22)])
def test_kernel_follows_the_step(ctx, d, hq, hkv, short, long):
    """Short steps run on the fp32 tiles (none at d = 256), long ones on the split tiles, also when
    the step changes between two calls of one layer configuration."""
    attn = Attention(hq, d, float(np.float32(d ** -0.5)), hkv, 0, 0)
    g = torch.Generator(device="cuda")
    g.manual_seed(d)
    arena = KvCacheArena(ctx, 1, 2, 16, hkv, d)
    ctx.set_timing(True)
    try:
        for n in [n for n in (short, long, short, long) if n]:
            q = torch.randn(n, hq, d, device="cuda", generator=g)
            k, v = torch.randn(2, n, hkv, d, device="cuda", generator=g)
            ctx.set(True, cu_seqlens_q=[0, n], cu_seqlens_k=[0, n], max_seqlen_q=n, max_seqlen_k=n)
            ctx.bind_kv_cache(arena)
            ctx.reset_stats()
            out = attn.forward(q, k, v, ctx)
            ctx.sync()
            fp32, _ = ctx.kernel_stats("prefill_fp32")
            split, _ = ctx.kernel_stats("prefill_split")
            assert (fp32, split) == ((1, 0) if n == short else (0, 1)), (n, fp32, split)
            assert torch.isfinite(out).all()
    finally:
        ctx.set_timing(False)
        ctx.clear()
        arena.close()
