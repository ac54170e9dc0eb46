"""o_proj tiles on split operands (three bf16 parts of every fp32 value) at magnitudes where a split
can go wrong: rows of x and W of unlike size, columns of x far above the ones that make the result,
the ends of the exponent range, infinities and NaN (taken again on fp32 instructions), zeros, and K
that ends inside a tile, against float64.

Bar: rel-L2 1e-5 of every output row, and of every output column, by itself.  Both sides add up to
2052 products in fp32; 2052 * 2^-24 = 1.2e-4 bounds any order, sqrt(2052) * 2^-24 = 2.7e-6 is what
independent roundings give."""

import numpy as np
import pytest
import torch

from gpu_checks import dev, say
from nanollvm_amd import Context, Linear

pytestmark = pytest.mark.gpu

# Rows x columns over one 32 x 32 block per CU, so the tiled kernel runs; ragged in both.
SHAPES = [(600, 260, 1000), (900, 64, 770), (1030, 2052, 300), (4500, 1028, 1000)]


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def data(rows, inf, outf, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, inf)).astype(np.float32)
    w = (rng.standard_normal((outf, inf)) / np.sqrt(inf)).astype(np.float32)
    return rng, x, w


def run(ctx, x, w, b=None):
    ctx.reset_stats()
    ctx.set_timing(True)
    y = Linear(dev(w), None if b is None else dev(b)).forward(dev(x), ctx)
    ctx.sync()
    launches, _ = ctx.kernel_stats("linear_tiles")
    ctx.set_timing(False)
    assert launches == 1, "the tiled kernel did not run"
    return y.cpu().numpy().astype(np.float64)


def exact(x, w):
    return (torch.from_numpy(x).double() @ torch.from_numpy(w).double().T.contiguous()).numpy()


def worst(got, want, axis):
    err = np.linalg.norm(got - want, axis=axis)
    size = np.linalg.norm(want, axis=axis)
    return float(np.max(err / np.where(size > 0, size, 1.0)))


@pytest.mark.parametrize("rows,inf,outf", SHAPES)
def test_rows_of_unlike_size(ctx, rows, inf, outf):
    rng, x, w = data(rows, inf, outf, rows)
    x *= np.exp2(rng.integers(-40, 41, (rows, 1))).astype(np.float32)
    w *= np.exp2(rng.integers(-40, 41, (outf, 1))).astype(np.float32)
    x[:, inf // 2:] *= np.float32(2.0 ** 12)  # scales rise half way through K
    x[5] = 0.0
    w[7] = 0.0
    got, want = run(ctx, x, w), exact(x, w)
    # Columns are compared at equal row sizes, rows at equal column sizes.
    rn = np.linalg.norm(x.astype(np.float64), axis=1, keepdims=True)
    cn = np.linalg.norm(w.astype(np.float64), axis=1)[None, :]
    rn[rn == 0], cn[cn == 0] = 1.0, 1.0
    g, e = got / rn / cn, want / rn / cn
    r = max(worst(g, e, 0), worst(g, e, 1))
    say(f"linear split {rows}x{inf}->{outf}: worst row or column rel_l2={r:.3e}")
    assert r <= 1e-5, r
    assert np.all(got[5] == 0.0) and np.all(got[:, 7] == 0.0)


@pytest.mark.parametrize("rows,inf,outf", SHAPES)
def test_infinities_and_nan(ctx, rows, inf, outf):
    rng, x, w = data(rows, inf, outf, rows + 1)
    b = rng.standard_normal(outf).astype(np.float32)
    x[3, inf - 1] = np.inf
    x[130, 0] = np.nan
    w[200, 1] = -np.inf
    got = run(ctx, x, w, b)
    with np.errstate(all="ignore"):
        want = exact(x, w) + b
    odd = ~np.isfinite(want)
    assert odd[3].all() and odd[130].all() and odd[:, 200].all()
    assert np.array_equal(got[odd], want[odd], equal_nan=True)
    got[odd] = want[odd] = 0.0
    assert worst(got, want, 1) <= 1e-5


@pytest.mark.parametrize("every", [0, 8, 2])
@pytest.mark.parametrize("bits", [20, 24, 30, 60])
@pytest.mark.parametrize("rows,inf,outf", SHAPES)
def test_columns_of_unlike_size(ctx, rows, inf, outf, bits, every):
    """x columns (the first, or every eighth or second) 2^bits above the others where W is 0: the
    result is made of the small ones alone."""
    _, x, w = data(rows, inf, outf, rows + 2)
    big = slice(0, 1) if every == 0 else slice(0, None, every)
    x[:, big] *= np.float32(2.0 ** bits)
    w[:, big] = 0.0
    got, want = run(ctx, x, w), exact(x, w)
    r = max(worst(got, want, 0), worst(got, want, 1))
    say(f"linear columns {rows}x{inf}->{outf} 2^{bits} every {every}: rel_l2={r:.3e}")
    assert r <= 1e-5, r


@pytest.mark.parametrize("rows,inf,outf", SHAPES)
def test_ends_of_the_exponent_range(ctx, rows, inf, outf):
    """Rows near the largest float with results far below it; sums of small products beside a
    large x element and a large W element that meet zeros."""
    _, x, w = data(rows, inf, outf, rows + 3)
    x[:, 0] = 1.0
    x[4] *= np.float32(2.0 ** 122)
    x[5] *= np.float32(2.0 ** 113)
    x[6] *= np.float32(2.0 ** -60)
    w[3] *= np.float32(2.0 ** -60)
    w[:, inf // 2] = 0.0
    x[6, inf // 2] = 2.0 ** 45
    x[:, inf - 1] = 0.0
    w[3, inf - 1] = 2.0 ** 45
    w[9] *= np.float32(2.0 ** -20)
    got, want = run(ctx, x, w), exact(x, w)
    assert np.all(np.isfinite(got))
    rn = np.linalg.norm(want, axis=1, keepdims=True)
    cn = np.linalg.norm(want / rn, axis=0, keepdims=True)
    r = max(worst(got / rn / cn, want / rn / cn, 0), worst(got / rn / cn, want / rn / cn, 1))
    say(f"linear ends {rows}x{inf}->{outf}: rel_l2={r:.3e}")
    assert r <= 1e-5, r
    assert abs(got[6, 3] - want[6, 3]) <= 1e-4 * abs(want[6, 3])


@pytest.mark.parametrize("rows,inf,outf", SHAPES)
def test_rows_near_the_smallest_float(ctx, rows, inf, outf):
    """Rows whose bits reach down to 2^-126 and below, where 16-bit parts no longer hold them."""
    _, x, w = data(rows, inf, outf, rows + 4)
    x *= np.exp2(-100.0 - np.arange(rows) % 20).astype(np.float32)[:, None]
    got, want = run(ctx, x, w), exact(x, w)
    r = worst(got, want, 1)
    say(f"linear smallest {rows}x{inf}->{outf}: rel_l2={r:.3e}")
    assert r <= 1e-5, r
