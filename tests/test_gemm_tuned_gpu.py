"""The rocBLAS solutions of the compiled-in table (gpt.c_amd/csrc/gemm_tuned.inc), through the entry points that run
them: each entry's problem as an sgemm or sgemm_strided_batched call, twice, against float64 on sampled rows.

The first call of a solution validates it and then runs it.  With beta = 0 the output starts as NaN (a solution must
not read it), otherwise as ones.  Bound: a chain of K fp32 products, 2-norm error of independent terms about
sqrt(K) 2^-25; 2e-5 x the largest output, as the other tests of rocBLAS products assert.
"""
import numpy as np
import pytest

from test_gemm_table import entries

pytestmark = pytest.mark.gpu


def pattern(n, seed):
    """n normal values, a block of 2^20 and a bit repeated (the largest operand has 4e8 values)."""
    block = np.random.default_rng(seed).standard_normal((1 << 20) + 7).astype(np.float32)
    return np.resize(block, n)


@pytest.mark.parametrize("key", [k for k, _ in entries()], ids=lambda k: "x".join(map(str, k[2:5])) + f"_{k[0]}{k[1]}_{k[11]}")
def test_table_solution(rt, key):
    # Column-major op(A) (m x k) op(B) (k x n) is the row-major C (n x m) = op(B)^T op(A)^T.
    ta, tb, m, n, k, lda, ldb, ldc, sa, sb, sc, batch, beta_zero, alpha_one = key
    print(f"case tuned {key}", flush=True)
    assert alpha_one
    nb = max(batch, 1)
    M, N, K, trans_a, trans_b = n, m, k, tb, ta
    rows_x, rows_w = (K if trans_a else M), (N if trans_b else K)
    X = pattern((nb - 1) * sb + rows_x * ldb, 1)
    W = pattern((nb - 1) * sa + rows_w * lda, 2)
    beta = 0.0 if beta_zero else 1.0
    C0 = np.full((nb - 1) * sc + M * ldc, np.nan if beta_zero else 1.0, np.float32)
    tx, tw, tc = rt.from_numpy(X), rt.from_numpy(W), rt.from_numpy(C0)
    pick = np.unique(np.linspace(0, M - 1, 23).astype(int))
    for call in range(2):
        if call == 1:
            rt.free(tc)
            tc = rt.from_numpy(C0)
        if batch:
            rt.lib.sgemm_strided_batched_cuda(trans_a, trans_b, M, N, K, 1.0, tx, ldb, sb, tw, lda, sa, beta, tc, ldc, sc, nb)
        else:
            rt.lib.sgemm_cuda(trans_a, trans_b, M, N, K, 1.0, tx, 0, ldb, tw, 0, lda, beta, tc, 0, ldc)
        got = rt.to_numpy(tc)
        for b in range(nb):
            x = X[b * sb:b * sb + rows_x * ldb].reshape(rows_x, ldb)
            w = W[b * sa:b * sa + rows_w * lda].reshape(rows_w, lda)[:, :K if trans_b else N].astype(np.float64)
            x = (x[:, pick].T if trans_a else x[pick, :K]).astype(np.float64)
            ref = x @ (w.T if trans_b else w) + beta
            err = np.abs(got[b * sc:b * sc + M * ldc].reshape(M, ldc)[pick, :N] - ref).max()
            assert err <= 2e-5 * np.abs(ref).max(), (b, err)
    for t in (tx, tw, tc):
        rt.free(t)
