"""Calls that take no scratch under graph capture: a replay must not write to blocks that the pool has handed on.

Each call runs eagerly first (its scratch, if it takes any, is then a block of the pool), is captured, and is replayed
several times between other work that owns every such block; each replay's outputs are the eager call's, and the
blocks' contents stay.
"""
import ctypes

import numpy as np
import pytest

import gptc

pytestmark = pytest.mark.gpu


class Graph:
    """What `call` launches on the library's stream, as a HIP graph."""

    def __init__(self, rt, call):
        self.hip = hip = ctypes.CDLL("libamdhip64.so")
        self.stream, graph, self.exec = ctypes.c_void_p(rt.stream()), ctypes.c_void_p(), ctypes.c_void_p()
        rt.sync()
        assert hip.hipStreamBeginCapture(self.stream, 1) == 0  # this thread's calls
        call()
        assert hip.hipStreamEndCapture(self.stream, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(self.exec), graph, None, None, ctypes.c_size_t(0)) == 0
        assert hip.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0

    def free(self):
        assert self.hip.hipGraphExecDestroy(self.exec) == 0


def slices(*floats):
    """The scratch sizes that slices of products of these sizes would take."""
    return [n * S for n in floats for S in range(2, 33 if n < 1 << 18 else 9)]


def replays_leave_the_pool_alone(rt, call, outputs, reset, scratch, tol):
    """scratch: floats of the blocks to hold; tol: the largest difference from the eager outputs, as a share of their
    largest value."""
    reset()
    call()
    eager = [rt.to_numpy(t) for t in outputs]
    graph = Graph(rt, call)
    held = [rt.empty((n,)) for n in scratch for _ in range(2)]
    for t in held:
        rt.lib.fill_tensor_data_cuda(t, ctypes.c_float(7.0))
    for _ in range(3):
        reset()
        rt.sync()
        graph.replay()
        rt.sync()
        for t, ref in zip(outputs, eager):
            assert np.abs(rt.to_numpy(t) - ref).max() <= tol * np.abs(ref).max()
        assert all((rt.to_numpy(t) == 7.0).all() for t in held)
    graph.free()
    for t in held:
        rt.free(t)


def rnd(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("rows,fin,fout", [(100, 768, 768), (64, 3072, 100)])
def test_linear_forward(rt, rows, fin, fout):
    """Reductions that the eager call cuts into slices."""
    print(f"case capture linear forward rows={rows} in={fin} out={fout}", flush=True)
    rng = np.random.default_rng(rows)
    x, W, b = (rt.from_numpy(v) for v in (rnd(rng, rows, fin), rnd(rng, fout, fin), rnd(rng, fout)))
    y = rt.empty((rows, fout))
    replays_leave_the_pool_alone(rt, lambda: rt.lib.linear_forward_cuda_kernel(W, b, x, y), [y],
                                 lambda: rt.lib.fill_tensor_data_cuda(y, ctypes.c_float(np.nan)),
                                 slices(rows * fout), 1e-6)
    for t in (x, W, b, y):
        rt.free(t)


@pytest.mark.parametrize("rows,fin,fout", [(1000, 777, 801), (640, 130, 8191)])
def test_linear_backward(rt, rows, fin, fout):
    print(f"case capture linear backward rows={rows} in={fin} out={fout}", flush=True)
    rng = np.random.default_rng(rows)
    x, W, g = (rt.from_numpy(v) for v in (rnd(rng, rows, fin), rnd(rng, fout, fin), rnd(rng, rows, fout)))
    dx, dW = rt.empty((rows, fin)), rt.empty((fout, fin))

    def reset():
        rt.lib.fill_tensor_data_cuda(dx, ctypes.c_float(np.nan))
        rt.lib.fill_tensor_data_cuda(dW, ctypes.c_float(0.0))

    replays_leave_the_pool_alone(rt, lambda: rt.lib.linear_backward_cuda_kernel(g, x, W, dW, None, dx), [dx, dW], reset,
                                 slices(rows * fin, fin * fout), 1e-6)
    for t in (x, W, g, dx, dW):
        rt.free(t)


@pytest.mark.parametrize("B,T,C,H", [(2, 129, 128, 2), (1, 1000, 192, 3)])
def test_attention_backward_with_qkv_bias(rt, B, T, C, H):
    """The column sums of the slab kernels (16 and 32 rows a slab) stay in the state."""
    print(f"case capture attention backward B={B} T={T} C={C} H={H}", flush=True)
    rng = np.random.default_rng(T)
    lib = rt.lib
    x, dy, bias = (rt.from_numpy(v) for v in (rnd(rng, B, T, 3 * C), rnd(rng, B, T, C), rnd(rng, 3 * C)))
    mask = rt.from_numpy(np.tril(np.ones((T, T), np.float32)))
    y, dout, db = rt.empty((B, T, C)), rt.empty((B, T, 3 * C)), rt.empty((3 * C,))
    caches = (gptc.TensorP * 4)(x, y, rt.empty((B, H, T)), rt.empty((int(lib.gptc_attention_state_floats(B, T, C, H)),)))
    lib.gptc_attention_forward_qkv_bias(x, bias, mask, H, caches, y)

    def reset():
        lib.fill_tensor_data_cuda(dout, ctypes.c_float(np.nan))
        lib.fill_tensor_data_cuda(db, ctypes.c_float(0.0))

    replays_leave_the_pool_alone(rt, lambda: lib.gptc_attention_backward_qkv_bias(dy, caches, bias, H, dout, db),
                                 [dout, db], reset, [B * ((T + r - 1) // r) * 3 * C for r in (16, 32)], 0)
    for t in (x, dy, bias, mask, y, dout, db, caches[2], caches[3]):
        rt.free(t)
