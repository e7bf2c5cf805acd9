"""GPU parity of gpt.c's model layers built on the library: the SelfAttention
block (qkv Linear -> fused attention -> c_proj) and the full GPT-2 training
step (forward, CrossEntropyLoss, backward, AdamW), driven through the same
C objects and call order as gpt.c's train_gpt.c:481-521, against the CPU
oracle's composition of gpt.c's CPU kernels (oracle/gpt2_oracle.py, pinned
against torch float64 autograd in tests/test_oracle_ops.py).

Tolerances: logits, loss and gradients within 1e-4 x max(1, max|ref|) per
tensor (fp32 GEMMs summed in different orders); parameters after each AdamW
step within 1e-5 x max(1, max|ref|).
"""
import numpy as np
import pytest

import gptc
from gpt2_oracle import GPT2Oracle, param_shapes

pytestmark = pytest.mark.gpu


def check(name, got, ref, rel=1e-4):
    ref = np.asarray(ref, np.float64)
    tol = rel * max(1.0, float(np.abs(ref).max()))
    err = float(np.abs(np.asarray(got, np.float64) - ref).max())
    print(f"  {name}: max abs err {err:.3e} (tol {tol:.1e})")
    assert np.isfinite(got).all(), name
    assert err <= tol, f"{name}: {err:.3e} > {tol:.1e}"


def init_params(V, block, L, C, seed, std=0.02):
    """C3's initialisation: N(0, std) matrices and embeddings, zero biases,
    LayerNorm weights 1 (biases 0)."""
    rng = np.random.default_rng(seed)
    out = []
    for name, shp in param_shapes(V, block, L, C):
        if name.endswith(("ln1.W", "ln2.W")) or name == "ln_f.W":
            out.append(np.ones(shp, np.float32))
        elif len(shp) == 1:
            out.append(np.zeros(shp, np.float32))
        else:
            out.append((rng.standard_normal(shp) * std).astype(np.float32))
    return out


def perturb_small(params, seed):
    """Non-trivial biases and LayerNorm parameters, so every gradient path is exercised."""
    rng = np.random.default_rng(seed)
    return [(p + 0.05 * rng.standard_normal(p.shape)).astype(np.float32) if p.ndim == 1 else p for p in params]


def gpu_train_steps(rt, params, batches, cfg, lr, wd, eps=1e-8):
    """train_gpt.c's loop on the GPU: zero_grad, forward, loss, backward, step.
    Returns per step (loss, logits, grads, params after the step)."""
    V, block, L, H, C = cfg
    model = gptc.GPT2Model(rt, block, V, L, H, C)
    model.fast_load(params)
    model.to(gptc.CUDA)
    opt = gptc.AdamWOptimizer(rt, model, lr=lr, beta1=0.9, beta2=0.99, eps=eps, weight_decay=wd)
    loss_fn = gptc.CrossEntropy(rt)
    out = []
    for ids, tg in batches:
        opt.zero_grad()
        x = rt.from_numpy(ids.astype(np.float32))
        t = rt.from_numpy(tg.astype(np.float32))
        logits = model.forward(x)
        losses = loss_fn.forward(logits, t)
        logits_np = rt.to_numpy(logits)
        rt.free(logits)
        B, T = ids.shape
        g = rt.from_numpy(np.ones((B, T), np.float32))
        g = loss_fn.backward(g)
        g = model.backward(g)
        if g:
            rt.free(g)
        grads = [rt.to_numpy(t_) for t_ in model.gradients()]
        opt.step()
        loss = float(rt.to_numpy(losses)[0])
        rt.free(losses)
        out.append((loss, logits_np, grads, [rt.to_numpy(p) for p in model.parameters()]))
    opt.free()
    loss_fn.free()
    model.free()
    return out


def oracle_train_steps(oracle, params, batches, L, H, lr, wd, eps=1e-8):
    g = GPT2Oracle(oracle, params, L, H)
    out = []
    for ids, tg in batches:
        logits = g.forward(ids)
        loss = g.loss(logits, tg)
        grads = g.backward()
        grads = [a.copy() for a in grads]
        g.step(lr=lr, weight_decay=wd, eps=eps)
        out.append((loss, logits, grads, [p.copy() for p in g.p]))
    return out


def compare_steps(names, gpu, ref):
    for s, ((lg, zg, gg, pg), (lr_, zr, gr, pr)) in enumerate(zip(gpu, ref)):
        print(f" step {s + 1}: loss gpu {lg:.6f} oracle {lr_:.6f}")
        assert abs(lg - lr_) <= 1e-4 * max(1.0, abs(lr_)), "loss"
        check(f"step {s + 1} logits", zg, zr)
        for n, a, b in zip(names, gg, gr):
            check(f"step {s + 1} grad {n}", a, b)
        for n, a, b in zip(names, pg, pr):
            check(f"step {s + 1} param {n}", a, b, rel=1e-5)


@pytest.mark.parametrize("V,block,L,H,C,B,T", [
    (97, 32, 2, 2, 64, 2, 32),        # tiny, head size 32
    (50257, 1024, 1, 12, 768, 2, 128),  # GPT-2 small's widths, one layer
    (211, 64, 3, 4, 96, 3, 40),       # ragged T (40 < block), D = 24
])
def test_gpt2_training_steps_match_oracle(rt, oracle, V, block, L, H, C, B, T):
    print(f"case gpt2 V={V} block={block} L={L} H={H} C={C} B={B} T={T}")
    rng = np.random.default_rng(V + T)
    params = perturb_small(init_params(V, block, L, C, seed=V), seed=C)
    batches = [(rng.integers(0, V, (B, T)), rng.integers(0, V, (B, T))) for _ in range(2)]
    # AdamW divides by sqrt(v) + eps: with gpt.c's eps = 1e-8 an entry whose
    # gradient is at rounding-noise level (1e-9) moves by up to lr either way,
    # so two correct implementations part by O(lr) there.  eps = 1e-4 keeps the
    # update Lipschitz in the gradient at this scale and the comparison strict
    # (eps = 1e-8 itself is exercised by the AdamW kernel test and C3 below).
    lr, wd, eps = 1e-3, 0.1, 1e-4
    gpu = gpu_train_steps(rt, params, batches, (V, block, L, H, C), lr, wd, eps)
    ref = oracle_train_steps(oracle, params, batches, L, H, lr, wd, eps)
    names = [n for n, _ in param_shapes(V, block, L, C)]
    compare_steps(names, gpu, ref)


@pytest.mark.parametrize("B,T,C,H", [
    (4, 256, 768, 12),  # GPT-2 small's widths: the qkv bias folded into the D = 64 kernels
    (2, 100, 256, 4),   # short heads (T <= 128): folded, P recomputed in dk/dv
    (1, 300, 128, 2),   # ragged T, folded
    (2, 77, 96, 4),     # D = 24: the bias is added to the qkv activations instead
    (2, 64, 256, 2),    # D = 128 (the 128-dim kernels), bias added to the activations
    (3, 65, 128, 2),    # two-tile heads with the bias folded into the short-head kernels
    (2, 50, 384, 2),    # D = 192 (the generic head-size kernels), bias added to the activations
])
def test_self_attention_block_matches_oracle(rt, oracle, B, T, C, H):
    """SelfAttention (self_attention.c:47-83): forward and backward through
    the library's layer objects vs the oracle's Linear -> attention -> Linear.
    On the GPU the layer folds the qkv Linear's bias into the attention
    kernels (and its gradient into their epilogues); the oracle adds it in
    the Linear, as gpt.c does."""
    self_attention_vs_oracle(rt, oracle, B, T, C, H)


@pytest.mark.parametrize("scratch", ["whole", "chunks", "none"])
@pytest.mark.parametrize("B,T,C,H", [(2, 256, 768, 12), (2, 100, 256, 4)])
def test_self_attention_lse_only_state(rt, oracle, B, T, C, H, scratch):
    """The same block with the attention state capped to the log-sum-exp: the
    bias folded into the recomputing dk/dv kernel and, with a dS scratch of
    every head ("whole") or of 5 heads at a time ("chunks"), into the dq
    kernel that reads it; with no scratch ("none"), dq's bias gradient comes
    from the recomputing dq kernel's column sums.  Shapes that run the slab
    backward need no scratch: tests/test_attention_tiled_gpu.py has the three
    modes for the others."""
    nqt = (T + 63) // 64
    limit = {"whole": -1, "chunks": 5 * nqt * (nqt + 1) * 2048, "none": 0}[scratch]
    rt.lib.gptc_attention_set_state_limit(0)
    rt.lib.gptc_attention_set_scratch_limit(limit)
    try:
        self_attention_vs_oracle(rt, oracle, B, T, C, H)
    finally:
        rt.lib.gptc_attention_set_state_limit(-1)
        rt.lib.gptc_attention_set_scratch_limit(-1)


def self_attention_vs_oracle(rt, oracle, B, T, C, H):
    import oracle as oracle_mod
    ops = oracle_mod.Ops(oracle)
    rng = np.random.default_rng(5 + T)
    Wq, bq = (rng.standard_normal((3 * C, C)) * 0.02).astype(np.float32), (rng.standard_normal(3 * C) * 0.1).astype(np.float32)
    Wp, bp = (rng.standard_normal((C, C)) * 0.02).astype(np.float32), (rng.standard_normal(C) * 0.1).astype(np.float32)
    x = rng.standard_normal((B, T, C)).astype(np.float32)
    g = rng.standard_normal((B, T, C)).astype(np.float32)
    sa = gptc.SelfAttentionBlock(rt, C, H, T, 1)
    sa.load_arrays([Wq, bq, Wp, bp])
    sa.to(gptc.CUDA)
    y = sa.forward(rt.from_numpy(x))
    y_np = rt.to_numpy(y)
    rt.free(y)
    dx = sa.backward(rt.from_numpy(g))
    dx_np = rt.to_numpy(dx)
    rt.free(dx)
    grads = [rt.to_numpy(t) for t in sa.gradients()]
    sa.free()
    qkv = ops.linear_forward(Wq, bq, x)
    a, q, k, v, att = oracle.forward(qkv, H)
    y_ref = ops.linear_forward(Wp, bp, a)
    dWp, dbp = np.zeros_like(Wp), np.zeros_like(bp)
    da = ops.linear_backward(g, a, Wp, dWp, dbp)
    dqkv = oracle.backward(da, H, q, k, v, att)
    dWq, dbq = np.zeros_like(Wq), np.zeros_like(bq)
    dx_ref = ops.linear_backward(dqkv, x, Wq, dWq, dbq)
    check("y", y_np, y_ref)
    check("dx", dx_np, dx_ref)
    for n, a_, b_ in zip(["dWqkv", "dbqkv", "dWproj", "dbproj"], grads, [dWq, dbq, dWp, dbp]):
        check(n, a_, b_)


@pytest.mark.parametrize("B", [1, 8])
def test_gpt2_c3_real_shape_matches_oracle(rt, oracle, B):
    """C3's model at its real width and depth (GPT-2 124M: 12 layers, C=768,
    H=12, V=50257, T=1024, N(0, 0.02) init, zero biases, LayerNorm weight 1),
    on a B=1 slice and at C3's own batch, B=8 (whose weight-gradient GEMMs
    reduce over 8192 rows, split four or eight ways into strided-batched
    slices): one training step against the oracle's step over the same
    batch, at gpt.c's AdamW eps = 1e-8.

    Loss, logits and all 148 gradient tensors within 1e-4 x max(1, max|ref|),
    and each gradient within D = 1e-3 x (its tensor's largest |ref|) + 1e-9.
    Parameters after the step: at step 1 AdamW moves each entry by
    u(g) = lr * g / (|g| + eps) (m-hat = g, v-hat = g^2, weight decay 0), so a
    gradient error d <= D moves the update by at most lr * eps * D / (|g| - D)^2
    where |g| > 2D, and by at most 2 lr where |g| <= 2D (there fp32 does not
    fix the update's sign).  Both bounds are asserted, plus the fp32 rounding
    of the update on either side (1e-6 lr + 2.4e-7 |p|); outside the tied
    embedding the second group must hold under 20 % of the entries (12 % at
    this init)."""
    V, block, L, H, C, T = 50257, 1024, 12, 12, 768, 1024
    print(f"case C3 real shape B={B} T={T}", flush=True)
    params = init_params(V, block, L, C, seed=2024)
    rng = np.random.default_rng(2025)
    batch = [(rng.integers(0, V, (B, T)), rng.integers(0, V, (B, T)))]
    lr, wd, eps = 3e-4, 0.0, 1e-8
    (lg, zg, gg, pg), = gpu_train_steps(rt, params, batch, (V, block, L, H, C), lr, wd, eps)
    (lr_, zr, gr, pr), = oracle_train_steps(oracle, params, batch, L, H, lr, wd, eps)
    names = [n for n, _ in param_shapes(V, block, L, C)]
    print(f"  loss gpu {lg:.6f} oracle {lr_:.6f}")
    assert abs(lg - lr_) <= 1e-4 * max(1.0, abs(lr_))
    check("logits", zg, zr)
    noisy = total = 0
    for n, g_gpu, g_ref, p0, p_gpu, p_ref in zip(names, gg, gr, params, pg, pr):
        check(f"grad {n}", g_gpu, g_ref)
        # A tighter per-tensor gradient bound for the step check: 1e-3 of the
        # tensor's largest gradient (asserted), so that "firm" covers the
        # entries whose update direction fp32 actually fixes.
        D = 1e-3 * float(np.abs(g_ref).max()) + 1e-9
        derr = float(np.abs(g_gpu.astype(np.float64) - g_ref).max())
        assert derr <= D, f"grad {n}: {derr:.3e} > 1e-3 of its largest entry ({D:.3e})"
        g = np.abs(g_ref.astype(np.float64))
        firm = g > 2 * D
        bound = np.where(firm, lr * eps * D / np.maximum(g - D, 1e-30) ** 2, 2 * lr)
        # fp32 evaluation on either side: u's bias corrections, sqrt, add and
        # divide (<= 8 roundings of 6e-8 each, so 1e-6 of lr |u| <= lr), and
        # the rounding of p - lr u (1.2e-7 of |p| per side).
        bound += 1e-6 * lr + 2.4e-7 * np.abs(p0.astype(np.float64))
        err = np.abs(p_gpu.astype(np.float64) - p_ref)
        assert (err <= bound).all(), f"param {n}: worst excess {float((err - bound).max()):.3e}"
        if n != "wte":
            noisy += int((~firm).sum())
            total += g.size
        print(f"    {n}: {int((~firm).sum())} of {g.size} entries with |grad| <= 2D")
    # wte is tied to lm_head: rows of tokens absent from the batch get only the
    # lm_head part of the gradient, far below the largest rows; they are left
    # out of the share.  Most of the rest are the q and k parts of the qkv
    # weights and biases, whose gradients at this init (near-uniform scores)
    # sit orders of magnitude below the v part's.
    print(f"  parameters within the AdamW bound; outside wte {noisy} of {total} entries have |grad| <= 2D")
    assert noisy < 0.2 * total


def test_gpt2_c3_full_size_step_properties(rt):
    """C3 at full size (GPT-2 124M, B=8, T=1024, N(0, 0.02) init): the step's
    size-independent properties -- the initial loss sits at ln V plus the
    logit variance term, everything is finite, the whole step is
    deterministic (two runs agree bit for bit), and one AdamW step lowers the
    loss on the same batch."""
    V, block, L, H, C, B, T = 50257, 1024, 12, 12, 768, 8, 1024
    params = init_params(V, block, L, C, seed=1337)
    rng = np.random.default_rng(1338)
    ids, tg = rng.integers(0, V, (B, T)), rng.integers(0, V, (B, T))
    runs = [gpu_train_steps(rt, params, [(ids, tg), (ids, tg)], (V, block, L, H, C), 3e-4, 0.0) for _ in range(2)]
    (l1, z1, g1, p1), (l2, _, _, _) = runs[0]
    print(f"  loss step 1 {l1:.6f}, step 2 (same batch) {l2:.6f}, ln V {np.log(V):.6f}")
    assert np.log(V) - 0.01 <= l1 <= np.log(V) + 0.5
    assert l2 < l1
    assert all(np.isfinite(a).all() for a in g1) and all(np.isfinite(a).all() for a in p1)
    (m1, y1, h1, q1), (m2, _, _, _) = runs[1]
    assert l1 == m1 and l2 == m2 and np.array_equal(z1, y1)
    assert all(np.array_equal(a, b) for a, b in zip(g1, h1)) and all(np.array_equal(a, b) for a, b in zip(p1, q1))
