"""GPU parity of the attention kernels on 64- and 128-row blocks where the slab kernels do not run: many heads at
ragged T, every state and scratch of the backward, with and without the qkv bias, and shapes whose forward runs one
kind and whose backward the other.  Each case asserts the route that it is here for (gptc_attention_slabs: bit 0 the
forward on slabs, bit 1 the backward); oracle and tolerance of tests/test_attention_gpu.py.
"""
import numpy as np
import pytest

from test_attention_gpu import compare_with_oracle, ds_floats_per_head, lse_only_state, qkv_inputs, run_layer, scratch_limit  # noqa: F401
from test_gpt2_gpu import self_attention_vs_oracle

pytestmark = pytest.mark.gpu


def check_route(rt, B, T, C, H, route):
    print(f"case route {route} B={B} T={T} C={C} H={H}", flush=True)
    assert rt.lib.gptc_attention_slabs(B, T, C, H) == route


@pytest.mark.parametrize("B,T,C,H,route", [
    (8, 333, 768, 12, 0), (10, 200, 768, 12, 0), (4, 1000, 768, 12, 0),   # heads of 64 with the stored P'
    (16, 100, 640, 10, 0), (25, 128, 704, 11, 0),                         # short heads
    (4, 333, 768, 12, 1), (2, 961, 768, 12, 1), (5, 200, 832, 13, 2),     # one direction on slabs
    (1, 1000, 1280, 20, 1),                                               # and key blocks cut in two
    (8, 200, 1536, 32, 0), (3, 1000, 960, 20, 0), (5, 333, 576, 24, 1),   # heads of 48 and 24
    (8, 200, 1536, 16, 0), (8, 333, 960, 12, 0), (2, 1000, 2560, 20, 0),  # of 96, 80 and 128
    (10, 97, 1280, 16, 0),
])
def test_tiled_against_oracle(rt, oracle, B, T, C, H, route):
    check_route(rt, B, T, C, H, route)
    compare_with_oracle(rt, oracle, B, T, C, H)


@pytest.mark.parametrize("scratch", ["whole", "chunks", "none"])
@pytest.mark.parametrize("B,T,C,H,route", [
    (2, 1000, 768, 12, 1), (6, 200, 1024, 16, 0), (4, 333, 768, 12, 1), (8, 333, 768, 12, 0), (16, 100, 640, 10, 0),
])
def test_tiled_lse_only_state(rt, oracle, lse_only_state, B, T, C, H, route, scratch):  # noqa: F811
    """The backward of the log-sum-exp-only state at ragged T, with the scratch of all heads, of 5 at a time (B H is no
    multiple of 5 but in the last) and none."""
    check_route(rt, B, T, C, H, route)
    with scratch_limit(rt, {"whole": -1, "chunks": 5 * ds_floats_per_head(T), "none": 0}[scratch]):
        compare_with_oracle(rt, oracle, B, T, C, H)


@pytest.mark.parametrize("B,T,C,H,route", [
    (8, 333, 768, 12, 0), (4, 333, 768, 12, 1), (5, 200, 832, 13, 2), (16, 100, 640, 10, 0), (1, 1000, 1280, 20, 1),
])
def test_tiled_with_qkv_bias(rt, oracle, B, T, C, H, route):
    """The bias folded into these kernels, and its gradient from their column sums."""
    check_route(rt, B, T, C, H, route)
    self_attention_vs_oracle(rt, oracle, B, T, C, H)


@pytest.mark.parametrize("scratch", ["whole", "chunks", "none"])
@pytest.mark.parametrize("B,T,C,H,route", [(6, 200, 1024, 16, 0), (4, 333, 768, 12, 1), (16, 100, 640, 10, 0)])
def test_tiled_lse_only_state_with_qkv_bias(rt, oracle, lse_only_state, B, T, C, H, route, scratch):  # noqa: F811
    check_route(rt, B, T, C, H, route)
    with scratch_limit(rt, {"whole": -1, "chunks": 5 * ds_floats_per_head(T), "none": 0}[scratch]):
        self_attention_vs_oracle(rt, oracle, B, T, C, H)


@pytest.mark.parametrize("T", [1000, 1024])
def test_split_key_blocks_run_and_repeat(rt, oracle, T):
    """20 heads fill 160 of the dk/dv kernel's 512 slots: key blocks run as two workgroups that add into dK, dV rows
    which the delta kernel zeroed.  Oracle parity, and the same bits again."""
    check_route(rt, 1, T, 1280, 20, 1)
    compare_with_oracle(rt, oracle, 1, T, 1280, 20)
    x, dy = qkv_inputs(rt, 1, T, 1280, 31, 32)
    first, second = (run_layer(rt, x, dy, 20) for _ in range(2))
    assert all(np.array_equal(a, b) for a, b in zip(first, second))
