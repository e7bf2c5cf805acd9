"""The Linear layers' products on the bf16 matrix cores (csrc/gemm_split.hip)
against float64 numpy, at the edges of their tiles and reductions.

Bound.  A step of 32 terms leaves out at most 3 x 2^-26 of each product and
rounds its sum twelve times (2^-23 of its size each, the matrix core's
truncation), and the steps' sums are added with K / 32 fp32 roundings:
|error| <= (2^-19 + (K / 32 + slices) 2^-24) sum |a||b| for each output, with at
most 32 slices.  The 2-norm error is held to 3e-7, under the 5e-7 and more
that a chain of fp32 sums shows from K = 768 on.
"""
import ctypes

import numpy as np
import pytest

import gptc

pytestmark = pytest.mark.gpu


def rnd(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


def check(name, got, a, b, add=0.0):
    """got = a @ b + add (float64 operands)."""
    K = a.shape[1]
    ref = a @ b + add
    tol = (2.0 ** -19 + (K / 32 + 32) * 2.0 ** -24) * (np.abs(a) @ np.abs(b) + np.abs(add)) + 1e-30
    err = np.abs(got - ref)
    rel = np.linalg.norm(err) / max(np.linalg.norm(ref), 1e-30)
    print(f"  {name}: 2-norm {rel:.2e}, largest share of the bound {(err / tol).max():.3f}")
    assert np.isfinite(got).all() and (err <= tol).all(), name
    assert rel <= 3e-7, name


class Case:
    """Device tensors, `shift` floats into their buffers (4-byte alignment only), outputs prefilled with NaN."""

    def __init__(self, rt, shift):
        self.rt, self.shift, self.owned = rt, shift, []

    def __call__(self, a):
        flat = np.concatenate([np.zeros(self.shift, np.float32), a.ravel()])
        t = self.rt.from_numpy(flat)
        self.owned.append(t)
        v = gptc.Tensor()
        ctypes.memmove(ctypes.byref(v), t, ctypes.sizeof(v))
        v.t = ctypes.cast(ctypes.cast(t.contents.t, ctypes.c_void_p).value + 4 * self.shift, ctypes.POINTER(ctypes.c_float))
        v.ndims, v.length = a.ndim, a.size
        for i, n in enumerate(a.shape):
            v.shape[i] = n
        return ctypes.pointer(v), t

    def get(self, pair, shape):
        return self.rt.to_numpy(pair[1])[self.shift:].reshape(shape).astype(np.float64)

    def free(self):
        for t in self.owned:
            self.rt.free(t)


@pytest.fixture
def case(rt):
    made = []

    def make(shift=0):
        made.append(Case(rt, shift))
        return made[-1]

    yield make
    for c in made:
        c.free()


def linear(rt, c, x, W, b, g):
    """y, dx, dW, db of one Linear; dW and db accumulate onto ones."""
    (rows, fin), fout = x.shape, W.shape[0]
    nan = lambda *s: np.full(s, np.nan, np.float32)  # noqa: E731
    tx, tW, tb, tg = c(x), c(W), c(b), c(g)
    y, dx, dW, db = c(nan(rows, fout)), c(nan(rows, fin)), c(np.ones((fout, fin), np.float32)), c(np.ones(fout, np.float32))
    rt.lib.linear_forward_cuda_kernel(tW[0], tb[0], tx[0], y[0])
    rt.lib.linear_backward_cuda_kernel(tg[0], tx[0], tW[0], dW[0], db[0], dx[0])
    return c.get(y, (rows, fout)), c.get(dx, (rows, fin)), c.get(dW, (fout, fin)), c.get(db, (fout,))


@pytest.mark.parametrize("rows,fin,fout,shift", [
    (1, 1, 1, 0), (64, 32, 64, 0), (65, 33, 63, 0), (3, 100, 77, 1), (130, 31, 129, 0), (200, 260, 300, 3),  # y only: the others are small
    (1000, 777, 801, 0),    # every product here, no size a multiple of anything
    (1000, 777, 801, 1),
    (2049, 640, 515, 0),    # one row past a tile
    (640, 130, 8191, 0),    # long sums for dx, cut into slices
    (70001, 96, 100, 0),    # long sums for dW, rows of 64-wide tiles
    (384, 1536, 1100, 2),
])
def test_linear_against_float64(rt, case, rows, fin, fout, shift):
    print(f"case linear rows={rows} in={fin} out={fout} shift={shift}", flush=True)
    rng = np.random.default_rng(rows + fin)
    x, W, b, g = rnd(rng, rows, fin), rnd(rng, fout, fin), rnd(rng, fout), rnd(rng, rows, fout)
    y, dx, dW, _ = linear(rt, case(shift), x, W, b, g)
    X, W64, G = (v.astype(np.float64) for v in (x, W, g))
    check("y", y, X, W64.T, b.astype(np.float64)[None, :])
    if rows * fin * fout >= 6e8:
        check("dx", dx, G, W64)
        check("dW", dW, G.T, X, 1.0)


@pytest.mark.parametrize("rows,fin,fout", [
    (1, 64, 4096), (8, 96, 50257), (33, 70, 8191), (130, 64, 16385),      # dx: long reductions
    (2048, 64, 64), (4096, 77, 30), (8192, 128, 96), (3000, 200, 60), (2050, 64, 33),  # dW: sliced, and rows that are not
    (2048, 512, 512),
])
def test_long_reductions_of_small_products(rt, case, rows, fin, fout):
    """Below the size at which every product runs here: dx over 4096 features and more does as well, and a weight
    gradient over 2048 rows and more is cut into slices of at least 1024 (2-norm error of a chain of K fp32 sums of
    independent terms: about sqrt(K) 2^-25, 8e-7 at the 1024 - 2047 rows of a slice; 2e-6 is asserted)."""
    print(f"case long rows={rows} in={fin} out={fout}", flush=True)
    rng = np.random.default_rng(rows + fout)
    x, W, b, g = rnd(rng, rows, fin), rnd(rng, fout, fin), rnd(rng, fout), rnd(rng, rows, fout)
    assert rows * fin * fout < 6e8
    _, dx, dW, _ = linear(rt, case(), x, W, b, g)
    X, W64, G = (v.astype(np.float64) for v in (x, W, g))
    if fout >= 4096:
        check("dx", dx, G, W64)
    ref = G.T @ X + 1.0
    rel = np.linalg.norm(dW - ref) / np.linalg.norm(ref)
    print(f"  dW: 2-norm {rel:.2e}")
    assert rel <= 2e-6


def test_outputs_are_not_shifted(rt, case):
    """The matrix core truncates towards minus infinity; the alternating signs of the steps cancel it.  The mean
    error over 8192 x 768 outputs is then a sample mean of errors of 2e-7 x the outputs' size: 1e-8 is 100 of its
    standard deviations, and half of the 4e-8 that K = 768 shows without the signs."""
    print("case shift", flush=True)
    rng = np.random.default_rng(5)
    rows, fin, fout = 8192, 768, 768
    x, W, b, g = rnd(rng, rows, fin), rnd(rng, fout, fin), np.zeros(fout, np.float32), rnd(rng, rows, fout)
    y, dx, _, _ = linear(rt, case(), x, W, b, g)
    X, W64, G = (v.astype(np.float64) for v in (x, W, g))
    for name, got, ref in (("y", y, X @ W64.T), ("dx", dx, G @ W64)):
        mean = (got - ref).mean() / np.sqrt((ref ** 2).mean())
        print(f"  {name}: mean error {mean:.2e} of the size")
        assert abs(mean) < 1e-8, name


@pytest.mark.parametrize("K", [7, 32, 96, 800])
def test_sums_of_odd_step_counts_are_not_shifted(rt, case, K):
    """One step, or an odd count of them, has no partner to cancel its truncation: the odd rows' and columns' signs
    do, in sums over either.  Independent errors give sums of them the relative size that the outputs' own errors
    have; twice that is asserted (a shift shows 8 to 17 times at K = 16 and 32, and 3 to 5 at 96)."""
    print(f"case odd steps K={K}", flush=True)
    rng = np.random.default_rng(K)
    rows, fout = 4096, 1024
    x, W, b, g = rnd(rng, rows, K), rnd(rng, fout, K), np.zeros(fout, np.float32), rnd(rng, rows, fout)
    y, _, _, _ = linear(rt, case(), x, W, b, g)
    ref = x.astype(np.float64) @ W.astype(np.float64).T
    err = y - ref
    own = np.linalg.norm(err) / np.linalg.norm(ref)
    for axis in (0, 1):
        share = np.linalg.norm(err.sum(axis)) / np.linalg.norm(ref.sum(axis)) / own
        print(f"  sums over axis {axis}: {share:.2f} of the outputs' error {own:.2e}")
        assert share < 2, axis


def test_infinities_and_large_values(rt, case):
    """An infinity (or a float that rounds up to one in bf16) splits into inf - inf; such blocks are formed again in
    fp32, so products that involve one are what fp32 gives, and all others stay exact to the bound."""
    print("case infinities", flush=True)
    rng = np.random.default_rng(6)
    rows, fin, fout = 900, 820, 840
    x, W, b, g = rnd(rng, rows, fin), rnd(rng, fout, fin), rnd(rng, fout), rnd(rng, rows, fout)
    W[W == 0] = 1.0
    x[3, 7], x[200, 1], x[899, 819] = np.inf, -np.inf, np.nan
    x[300, 5] = np.float32(3.4e38)                        # past the largest bf16
    W[:, 5] = np.where(np.arange(fout) % 2, 0.5, -0.25)   # its products stay finite
    y, _, dW, _ = linear(rt, case(), x, W, b, g)
    ref = x.astype(np.float64) @ W.astype(np.float64).T + b
    bad = {3, 200, 899}
    for r in bad:
        assert np.array_equal(np.isnan(y[r]), np.isnan(ref[r])) and np.array_equal(y[r] > 0, ref[r] > 0), r
        assert not np.isfinite(y[r]).any()
    assert np.allclose(y[300], ref[300], rtol=1e-6)
    rest = [r for r in range(rows) if r not in bad | {300}]
    check("y, other rows", y[rest], x[rest].astype(np.float64), W.astype(np.float64).T, b.astype(np.float64)[None, :])
    cols = [c for c in range(fin) if c not in (7, 1, 819, 5)]
    check("dW, other columns", dW[:, cols], g.astype(np.float64).T, x[:, cols].astype(np.float64), 1.0)
    assert not np.isfinite(dW[:, [7, 1, 819]]).any()


@pytest.mark.parametrize("ex,ew", [(-114, 60), (-118, 60), (-125, 90), (60, -114), (90, -125), (-60, -60)])
def test_tiny_operands_keep_their_bits(rt, case, ex, ew):
    """Normal floats down to the smallest keep all 24 bits (bf16 has nothing below 2^-133, so unscaled parts of floats
    below 2^-110 would lose them); values of 2^ex times ordinary ones against 2^ew, the same bound as elsewhere."""
    print(f"case tiny ex={ex} ew={ew}", flush=True)
    rng = np.random.default_rng(7)
    rows, fin, fout = 1000, 1201, 1100
    scale = lambda a, e: np.ldexp(np.where(np.abs(a) < 1, np.copysign(np.float32(1), a), a), e).astype(np.float32)  # noqa: E731
    x, W, g = scale(rnd(rng, rows, fin), ex), scale(rnd(rng, fout, fin), ew), scale(rnd(rng, rows, fout), ex)
    y, dx, _, _ = linear(rt, case(), x, W, np.zeros(fout, np.float32), g)
    X, W64, G = (np.ldexp(v.astype(np.float64), -e) for v, e in ((x, ex), (W, ew), (g, ex)))
    check("y", np.ldexp(y, -ex - ew), X, W64.T)
    check("dx", np.ldexp(dx, -ex - ew), G, W64)
    # dW: g of 2^ex against x of 2^ew, onto zeros
    x2 = scale(rnd(rng, rows, fin), ew)
    c = case()
    tg, tx, tW = c(g), c(x2), c(W)
    dW, db, dx2 = c(np.zeros((fout, fin), np.float32)), c(np.zeros(fout, np.float32)), c(np.zeros((rows, fin), np.float32))
    rt.lib.linear_backward_cuda_kernel(tg[0], tx[0], tW[0], dW[0], db[0], dx2[0])
    check("dW", np.ldexp(c.get(dW, (fout, fin)), -ex - ew), G.T, np.ldexp(x2.astype(np.float64), -ew))


@pytest.mark.parametrize("ex,ew", [(70, 40), (105, -60), (-60, 105), (40, 40)])
def test_large_operands_and_sums(rt, case, ex, ew):
    """Floats past 2^104 and sums past 2^80 overflow the split's scale: those blocks are formed in fp32 instead, finite
    and within what a chain of K fp32 sums shows (2-norm about sqrt(K) 2^-25, 1e-6 here; 2e-6 is asserted)."""
    print(f"case large ex={ex} ew={ew}", flush=True)
    rng = np.random.default_rng(8)
    rows, fin, fout = 1000, 777, 801
    x, W, g = (np.ldexp(rnd(rng, *s), e) for s, e in (((rows, fin), ex), ((fout, fin), ew), ((rows, fout), ex)))
    y, dx, _, _ = linear(rt, case(), x, W, np.zeros(fout, np.float32), g)
    X, W64, G = (np.ldexp(v.astype(np.float64), -e) for v, e in ((x, ex), (W, ew), (g, ex)))
    for name, got, ref in (("y", y, X @ W64.T), ("dx", dx, G @ W64)):
        rel = np.linalg.norm(np.ldexp(got, -ex - ew) - ref) / np.linalg.norm(ref)
        print(f"  {name}: 2-norm {rel:.2e}")
        assert np.isfinite(got).all() and rel <= 2e-6, name
