"""GPU parity of the slab kernels (csrc/attn_slab.hip) at the edges of their
blocks, slabs and tiles, against the oracle at the tolerance of
tests/test_attention_gpu.py, for one and two row blocks per wave, every padded
head size, and the qkv bias folded in.
"""
import ctypes

import numpy as np
import pytest

import gptc
from test_attention_gpu import check, compare_with_oracle, lse_fp64, qkv_inputs
from test_gpt2_gpu import self_attention_vs_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,C,H", [
    # heads of 64: one block per slab (few tiles), T around blocks, slabs and tiles
    (1, 15, 64, 1), (1, 16, 64, 1), (2, 17, 128, 2), (1, 64, 128, 2), (1, 65, 128, 2), (2, 128, 256, 4),
    (1, 129, 64, 1), (1, 143, 128, 2), (1, 144, 64, 1), (1, 145, 64, 1), (2, 192, 128, 2), (1, 193, 64, 1),
    (1, 321, 192, 3),
    # two blocks per slab (350 tiles or more)
    # (their forward runs the tiled kernels at T = 176 to 191)
    (5, 176, 768, 12), (5, 177, 768, 12), (5, 191, 768, 12), (1, 1024, 192, 3), (1, 1009, 192, 3),
    # other head sizes: 4, 16, 36, 60 padded to 64, and 68, 80, 124, 128 to 128
    (2, 33, 8, 2), (1, 100, 16, 1), (2, 70, 72, 2), (3, 200, 120, 2), (2, 48, 136, 2), (2, 161, 160, 2), (1, 97, 248, 2),
    (1, 640, 512, 4), (8, 200, 512, 4), (2, 512, 96, 3),
    (1, 1009, 1024, 8), (1, 1000, 768, 8),  # from 1000 tiles on heads past 64 run two blocks forward too
])
def test_slabs_against_oracle(rt, oracle, B, T, C, H):
    print(f"case slab B={B} T={T} C={C} H={H}", flush=True)
    assert rt.lib.gptc_attention_slabs(B, T, C, H) & 2
    compare_with_oracle(rt, oracle, B, T, C, H)


@pytest.mark.parametrize("B,T,C,H", [(1, 40, 128, 2), (2, 129, 128, 2), (1, 333, 192, 3), (5, 177, 768, 12), (1, 1009, 192, 3)])
def test_slabs_with_qkv_bias(rt, oracle, B, T, C, H):
    """The bias added to the rows and its gradient from the slabs' column sums (one and two blocks per slab)."""
    print(f"case slab bias B={B} T={T} C={C} H={H}", flush=True)
    assert rt.lib.gptc_attention_slabs(B, T, C, H) & 2
    self_attention_vs_oracle(rt, oracle, B, T, C, H)


@pytest.mark.parametrize("B,T,C,H", [
    (1, 15, 64, 1), (1, 40, 128, 2), (2, 129, 128, 2), (3, 333, 192, 3),          # one block per slab
    (1, 1009, 192, 3), (4, 200, 512, 8), (1, 640, 448, 7), (3, 321, 448, 7),      # two (350 tiles or more)
])
def test_slabs_with_a_large_qkv_bias(rt, oracle, B, T, C, H):
    """Biases of the rows' own size through the entry points: y, the log-sum-exp, dqkv and db against the oracle on
    the rows with the bias added, one backward of a head's q, k and v parts each."""
    print(f"case slab large bias B={B} T={T} C={C} H={H}", flush=True)
    x, dy = qkv_inputs(rt, B, T, C)
    bias = rt.normal((3 * C,), 5)
    lib = rt.lib
    xt, dyt, bt = rt.from_numpy(x), rt.from_numpy(dy), rt.from_numpy(bias)
    mask = rt.from_numpy(np.tril(np.ones((T, T), np.float32)))
    yt, dout, db = rt.empty((B, T, C)), rt.empty((B, T, 3 * C)), rt.from_numpy(np.zeros(3 * C, np.float32))
    caches = (gptc.TensorP * 4)(xt, yt, rt.empty((B, H, T)), rt.empty((int(lib.gptc_attention_state_floats(B, T, C, H)),)))
    lib.gptc_attention_forward_qkv_bias(xt, bt, mask, H, caches, yt)
    lib.gptc_attention_backward_qkv_bias(dyt, caches, bt, H, dout, db)
    y, lse, d, dbias = rt.to_numpy(yt), rt.to_numpy(caches[2]), rt.to_numpy(dout), rt.to_numpy(db)
    for t in (xt, dyt, bt, mask, yt, dout, db, caches[2], caches[3]):
        rt.free(t)
    y_ref, q, k, v, att = oracle.forward(x + bias, H)
    d_ref = oracle.backward(dy, H, q, k, v, att)
    check("y", y, y_ref)
    check("lse", lse.reshape(B, H, T), lse_fp64(q, k))
    check("dqkv", d, d_ref)
    # Column sums of B T rows, each within the rows' own tolerance of independent sign.
    check("db", dbias, d_ref.astype(np.float64).sum((0, 1)), 1e-4 * np.sqrt(B * T))


def test_slabs_are_deterministic(rt):
    """The waves' partial results join in wave order: the same bits on every run."""
    B, T, C, H = 3, 333, 320, 5
    x, dy = rt.normal((B, T, 3 * C), 11), rt.normal((B, T, C), 12)
    seen = []
    for _ in range(2):
        layer = gptc.AttentionLayer(rt, C, H, T)
        layer.to(gptc.CUDA)
        y = layer.forward(rt.from_numpy(x))
        y_np = rt.to_numpy(y)
        d = layer.backward(rt.from_numpy(dy))
        seen.append((y_np, rt.to_numpy(d)))
        rt.free(y)
        rt.free(d)
        layer.free()
    assert all(np.array_equal(a, b) for a, b in zip(*seen))


def shifted(rt, shape, shift):
    """A tensor `shift` floats into a buffer (4-byte alignment only), and the buffer."""
    n = int(np.prod(shape))
    buf = rt.empty((n + shift,))
    v = gptc.Tensor()
    ctypes.memmove(ctypes.byref(v), buf, ctypes.sizeof(v))
    v.t = ctypes.cast(ctypes.cast(buf.contents.t, ctypes.c_void_p).value + 4 * shift, ctypes.POINTER(ctypes.c_float))
    v.ndims, v.length = len(shape), n
    for i, d in enumerate(shape):
        v.shape[i] = d
    return ctypes.pointer(v), buf


def prefilled_state_vs_oracle(rt, oracle, B, T, C, H, shift):
    """Forward into a state that is NaN throughout, then backward into gradients `shift` floats into their buffer."""
    x, dy = qkv_inputs(rt, B, T, C)
    lib = rt.lib
    xt, dyt = rt.from_numpy(x), rt.from_numpy(dy)
    mask = rt.from_numpy(np.tril(np.ones((T, T), np.float32)))
    state = rt.empty((int(lib.gptc_attention_state_floats(B, T, C, H)),))
    lib.fill_tensor_data_cuda(state, ctypes.c_float(np.nan))
    yt = rt.empty((B, T, C))
    caches = (gptc.TensorP * 4)(xt, yt, rt.empty((B, H, T)), state)
    lib.attention_forward_cuda_kernel(xt, mask, H, caches, yt)
    y = rt.to_numpy(yt)
    dout, buf = shifted(rt, (B, T, 3 * C), shift)
    lib.attention_backward_cuda_kernel(dyt, caches, H, dout)
    d = rt.to_numpy(buf)[shift:].reshape(B, T, 3 * C)
    for t in (xt, dyt, mask, yt, buf, caches[2], caches[3]):
        rt.free(t)
    y_ref, q, k, v, att = oracle.forward(x, H)
    check("y", y, y_ref)
    check("dqkv", d, oracle.backward(dy, H, q, k, v, att))


@pytest.mark.parametrize("B,T,C,H,shift", [
    (4, 333, 768, 12, 0), (2, 1000, 768, 12, 0), (1, 650, 1600, 25, 0),   # heads of 64
    (2, 1000, 1056, 22, 0), (5, 200, 480, 30, 0),                         # of 48 and 16
    (5, 333, 1152, 12, 0), (5, 200, 1920, 15, 0),                         # of 96 and 128
    (2, 140, 128, 2, 1), (1, 333, 96, 2, 1), (1, 70, 256, 2, 1),          # gradients that are not 16-byte aligned
])
def test_stored_probabilities_past_the_last_row(rt, oracle, B, T, C, H, shift):
    """A backward that the slabs do not serve reads the forward's P' in halves of 32 queries, rows past T among them
    that a slab of 16 rows does not write (T ends in the first 16 rows of a half here).  The state is NaN before the
    forward: those rows must not reach dK and dV as 0 * NaN."""
    print(f"case halves B={B} T={T} C={C} H={H} shift={shift}", flush=True)
    assert 0 < T % 32 <= 16 and (shift or rt.lib.gptc_attention_slabs(B, T, C, H) == 1)
    prefilled_state_vs_oracle(rt, oracle, B, T, C, H, shift)


@pytest.mark.parametrize("B,T,C,H", [(2, 17, 192, 3), (1, 64, 64, 1), (2, 100, 256, 4), (1, 128, 128, 2)])
def test_unaligned_gradients_of_short_heads(rt, oracle, B, T, C, H):
    """Heads of 64 up to 128 rows keep no P': the backward into gradients without 16-byte rows recomputes it too."""
    print(f"case short unaligned B={B} T={T} C={C} H={H}", flush=True)
    prefilled_state_vs_oracle(rt, oracle, B, T, C, H, 1)
