"""The residual forms (Linear forward + add, LayerNorm backward + add) against the
plain entry points followed by the addition, in numpy.

Bounds.  The LayerNorm's terms are the same sum with one more fp32 addition; the
two forms may contract a different product into an fma, which moves each of the
at most eight roundings: 2^-20 of the sum of the terms' sizes covers them.  The
Linear's term joins a sum of K products: 2-norm error against float64 under 3e-7
on the matrix-core path, and 2e-5 x the largest output on the other (add in place,
no bias, and smaller than where the split pays).
"""
import numpy as np
import pytest

import gptc

pytestmark = pytest.mark.gpu


def rnd(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("rows,fin,fout,bias", [
    (1, 64, 48, True), (3, 100, 77, True), (65, 33, 63, False), (129, 256, 130, True), (1000, 777, 801, False),
])
@pytest.mark.parametrize("in_place", [False, True])
def test_linear_forward_add(rt, rows, fin, fout, bias, in_place):
    print(f"case linear add rows={rows} in={fin} out={fout} bias={bias} in_place={in_place}", flush=True)
    rng = np.random.default_rng(rows + fout)
    x, W, b, a = rnd(rng, rows, fin), rnd(rng, fout, fin), rnd(rng, fout), rnd(rng, rows, fout)
    tx, tW, tb, ta = (rt.from_numpy(v) for v in (x, W, b, a))
    ty = ta if in_place else rt.from_numpy(np.full_like(a, np.nan))
    rt.lib.gptc_linear_forward_add_cuda(tW, tb if bias else None, tx, ta, ty)
    got, kept = rt.to_numpy(ty).astype(np.float64), rt.to_numpy(ta)
    for t in {id(t): t for t in (tx, tW, tb, ta, ty)}.values():
        rt.free(t)
    ref = x.astype(np.float64) @ W.astype(np.float64).T + a + (b if bias else 0)
    assert in_place or np.array_equal(kept, a)
    assert np.abs(got - ref).max() <= 2e-5 * np.abs(ref).max()
    if bias or not in_place or rows * fin * fout >= 6e8:
        assert np.linalg.norm(got - ref) <= 3e-7 * np.linalg.norm(ref)


# 5: the kernel of single columns; 2048: the widest; 1 row and rows that do not fill a workgroup's share
@pytest.mark.parametrize("rows,C", [(1, 768), (14, 5), (65, 768), (33, 1600), (3, 2048), (20000, 64)])
def test_layer_norm_backward_add(rt, rows, C):
    print(f"case layer_norm add rows={rows} C={C}", flush=True)
    rng = np.random.default_rng(rows + C)
    x, g, a, W = rnd(rng, rows, C), rnd(rng, rows, C), rnd(rng, rows, C), rnd(rng, C)
    mean, rstd = x.mean(1), 1 / np.sqrt(x.var(1) + np.float32(1e-5))
    zero = np.zeros(C, np.float32)
    tg, tW, ta, tx, tm, tr, dW, db, dW2, db2 = (rt.from_numpy(v) for v in (g, W, a, x, mean, rstd, zero, zero, zero, zero))
    out, dx = (rt.from_numpy(np.full_like(x, np.nan)) for _ in range(2))
    cache = (gptc.TensorP * 3)(tm, tr, tx)
    rt.lib.gptc_layer_norm_backward_add(tg, cache, tW, dW, db, ta, out)
    rt.lib.gptc_layer_norm_backward_set(tg, cache, tW, dW2, db2, dx)
    vals = [rt.to_numpy(t) for t in (out, dx, ta, dW, dW2, db, db2)]
    for t in (tg, tW, ta, tx, tm, tr, dW, db, dW2, db2, out, dx):
        rt.free(t)
    got, plain, kept, w1, w2, b1, b2 = vals
    gw, xhat = np.abs(g * W), np.abs((x - mean[:, None]) * rstd[:, None])
    size = np.abs(a) + rstd[:, None] * (gw + gw.mean(1, keepdims=True) * (1 + xhat * xhat.max(1, keepdims=True)))
    assert np.array_equal(kept, a) and (np.abs(got - (a + plain)) <= 2.0 ** -20 * size).all()
    assert np.array_equal(w1, w2) and np.array_equal(b1, b2)
    s = np.abs(g).sum(0, dtype=np.float64)  # a chain of at most 128 fp32 sums of these
    assert (np.abs(b1 - g.sum(0, dtype=np.float64)) <= 128 * 2.0 ** -24 * s).all()
