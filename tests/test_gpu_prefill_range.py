"""Prefill where one key, V row or V channel dwarfs what the result is made of.

The split kernel holds probabilities and V in fp16 parts beside a power of two, so their steps are
fixed beside the largest value in their units.  Here most of the weight (or the largest |v|) sits
where it adds nothing to the result: a sink key with no V, a V row that no query weighs, V tiles
of unlike size, a V channel far above the others.  Each query row of each head is compared with
float64 by itself (channels of unlike size by themselves).

Bar: 4e-6.  Up to 4096 fp32 products per output give sqrt(4096) * 2^-24 = 3.8e-6 if their
roundings are independent.  (The fp32 tiles reach 0.6e-6 to 7e-6 on these inputs.)"""

import numpy as np
import pytest
import torch

from cases import Case
from gpu_checks import dev, load_arena, say
from nanollvm_amd import Attention, Context
from nanollvm_amd import workloads as W
from test_gpu_prefill_split import exact

pytestmark = pytest.mark.gpu

BAR = 4e-6
N = 4096
HEADS = [(64, 1), (64, 4), (128, 2), (256, 4), (512, 2)]


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def build(d, rep, seed, seqs=((0, N), (0, 77), (0, 5), (0, 13))):
    rng = np.random.default_rng(seed)
    wl = W.build(f"range d{d} rep{rep}", list(seqs), is_prefill=True, hq=2 * rep, hkv=2, d=d,
                 scale=float(np.float32(d ** -0.5)), rng=rng, block_size=256, pool_cap=20000)
    case = Case(wl, seed=seed)
    # Dim 0 sets the score of single keys: every query has the same 4 there, the keys 0.
    case.q[:, :, 0] = 4.0
    case.k[:, :, 0] = 0.0
    return case


def set_score(case, key, score):
    case.k[key] = 0.0
    case.k[key, :, 0] = score / (4.0 * case.wl.scale)


def sink_score(weight, keys):
    """Score that takes this share of the softmax beside `keys` others of score N(0, 1)."""
    return np.log(weight / (1.0 - weight) * keys) + 0.5


def check(ctx, case, name, channels=slice(None), rows=slice(None), bar=BAR,
          mean=False):
    wl, m = case.wl, case.wl.meta
    say(name)
    arena = load_arena(ctx, case)
    try:
        ctx.set(**m.context_args())
        ctx.bind_kv_cache(arena)
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
    kc, vc = case.k_cache.copy(), case.v_cache.copy()
    slots = np.asarray(m.slot_mapping, np.int64)
    kc.reshape(-1, wl.hkv, wl.d)[slots] = case.k
    vc.reshape(-1, wl.hkv, wl.d)[slots] = case.v
    want = exact(case, kc, vc)
    assert np.all(np.isfinite(got))
    err = np.linalg.norm((got - want)[rows][..., channels], axis=-1)
    size = np.linalg.norm(want[rows][..., channels], axis=-1)
    rel = err / np.where(size > 0, size, 1.0)
    rel = float(np.mean(rel) if mean else np.max(rel))
    say(f"{name}: {'mean' if mean else 'worst'} row rel_l2={rel:.3e}")
    assert rel <= bar, rel


@pytest.mark.parametrize("v", [0.0, 1e-3])
@pytest.mark.parametrize("weight", [0.7, 0.98, 0.9995])
@pytest.mark.parametrize("d,rep", HEADS)
def test_sink_key(ctx, d, rep, weight, v):
    """The first key takes most of the weight (of the last row; more of the earlier ones) and adds
    little or nothing."""
    case = build(d, rep, seed=11)
    set_score(case, 0, sink_score(weight, N))
    case.v[0] *= np.float32(v)
    check(ctx, case, f"sink d{d} rep{rep} weight {weight} v {v}")


@pytest.mark.parametrize("factor", [2.0 ** 10, 2.0 ** 12, 8000.0, 2.0 ** 20])
@pytest.mark.parametrize("d,rep", HEADS)
def test_v_row_without_weight(ctx, d, rep, factor):
    """Most of the weight on one key, and beside it a large V row that no query weighs."""
    case = build(d, rep, seed=12)
    set_score(case, 5, sink_score(0.64, N))
    set_score(case, 40, -60.0)
    case.v[40] *= np.float32(factor)
    check(ctx, case, f"v row d{d} rep{rep} factor {factor}")


@pytest.mark.parametrize("span", [8, 14])
@pytest.mark.parametrize("d,rep", HEADS)
def test_v_tiles_of_unlike_size(ctx, d, rep, span):
    """V over 2^-span .. 2^0 by tiles of 32 keys; the weight on a row of the smallest."""
    case = build(d, rep, seed=13)
    t = np.arange(case.wl.tokens) // 32
    case.v *= np.exp2(-((t * 5) % (span + 1))).astype(np.float32)[:, None, None]
    small = 32 * int(np.argmax((t[::32] * 5) % (span + 1) == span))
    set_score(case, small + 3, sink_score(1.0 - 2.0 ** -(span + 1), N))
    check(ctx, case, f"v tiles d{d} rep{rep} span {span}")


@pytest.mark.parametrize("bits", [12, 20, 24, 30])
@pytest.mark.parametrize("d,rep", HEADS)
def test_v_channel(ctx, d, rep, bits):
    """One V channel 2^bits above the others, which are compared without it."""
    case = build(d, rep, seed=14)
    case.v[:, :, 5] *= np.float32(2.0 ** bits)
    check(ctx, case, f"v channel d{d} rep{rep} 2^{bits}", channels=np.r_[:5, 6:d])


@pytest.mark.parametrize("bits", [8, 12, 13, 14, 15, 17])
@pytest.mark.parametrize("d,rep", HEADS)
def test_k_channel(ctx, d, rep, bits):
    """One K channel 2^bits above the others where q is 0, so that no score shows it: the rows of a
    few keys, where a score's error shows most.  Bar: 3 sqrt(32) * 2^-24."""
    case = build(d, rep, seed=15)
    case.q[:, :, 5] = 0.0
    case.k[:, :, 5] *= np.float32(2.0 ** bits)
    check(ctx, case, f"k channel d{d} rep{rep} 2^{bits}", rows=slice(0, 32), bar=1e-6)


@pytest.mark.parametrize("d,rep", HEADS)
def test_zero_dims(ctx, d, rep):
    """Half of V's dims zero (at d = 256 and 512 those of whole waves), and keys without any V."""
    case = build(d, rep, seed=16)
    case.v[:, :, d // 2:] = 0.0
    case.v[100:400] = 0.0
    check(ctx, case, f"zero dims d{d} rep{rep}")


@pytest.mark.parametrize("d,rep", HEADS)
def test_few_keys(ctx, d, rep):
    """Rows of up to 32 keys, all of one tile: the probabilities' own rounding shows.  Bar, for the
    mean row: 1.9e-7, between what the products leave (1.5e-7 to 1.75e-7) and that with another
    2^-22 in the argument of every probability near 1, as beside a term of 8 to 16 (2.0e-7 to
    2.3e-7)."""
    case = build(d, rep, seed=17)
    check(ctx, case, f"few keys d{d} rep{rep}", rows=slice(1, 32), bar=1.9e-7, mean=True)


@pytest.mark.parametrize("seed", range(24))
def test_random_magnitudes(ctx, seed):
    """Steps with several of these at once, by chance: V rows, channels and tiles over up to 2^30, a
    few rows far above the others, zero channels, sharper scores, K channels that no score shows,
    keys with most of the weight.  Bar: 1e-5, the attention bar; on twenty times as many seeds the
    worst row was 7.2e-6 off, on the fp32 tiles 1.1e-5."""
    rng = np.random.default_rng(1000 + seed)
    d = int(rng.choice([64, 128, 256, 512]))
    case = build(d, int(rng.choice([1, 2, 4])), seed=1000 + seed,
                 seqs=((0, 1100 if d == 512 else 2100), (int(rng.integers(1, 400)), 90)))
    T, N, what = case.wl.tokens, case.wl.seqs[0][1], []

    def chance(p, name):
        what.append(name if rng.random() < p else "")
        return what[-1] != ""

    def spread(bits, shape):
        return np.exp2(rng.uniform(-bits, 0, shape)).astype(np.float32)

    if chance(0.4, "rows"):
        case.v *= spread(rng.uniform(0, 30), (T, 1, 1))
    if chance(0.4, "channels"):
        case.v *= spread(rng.uniform(0, 30), (1, 1, d))
    if chance(0.3, "tiles"):
        case.v *= np.exp2(-(np.arange(T) // 32 * int(rng.integers(1, 9)) % 20)).astype(
            np.float32)[:, None, None]
    if chance(0.3, "outliers"):
        case.v[rng.integers(0, T, 5)] *= np.float32(2.0 ** rng.uniform(0, 25))
    if chance(0.3, "zeros"):
        case.v[:, :, rng.random(d) < 0.3] = 0.0
    if chance(0.3, "sharp"):
        case.q[:, :, 1:] *= np.float32(2.0 ** rng.uniform(0, 3))
    if chance(0.3, "k channel"):
        case.k[:, :, 7] *= np.float32(2.0 ** rng.uniform(0, 16))
        case.q[:, :, 7] = 0.0
    if chance(0.5, "sinks"):
        for key in [0] if rng.random() < 0.5 else rng.integers(0, N, 3):
            set_score(case, key, rng.uniform(2, 25))
            case.v[key] *= np.float32(rng.choice([0.0, 1e-4, 1e-2, 1.0, 100.0]))
    check(ctx, case, f"random {seed} d{d}: {' '.join(w for w in what if w)}", bar=1e-5)
