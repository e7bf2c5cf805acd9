"""Which kernels a shape's attention runs (gptc_attention_slabs; csrc/attn_slab.hip): the rule on the host, no GPU.

Bit 0: the forward runs the slab kernels, bit 1: the backward.
"""
import pytest


@pytest.mark.parametrize("B,T,C,H,route", [
    (2, 100, 256, 4, 2),       # heads of 64 up to 128 rows: the short-head forward
    (8, 128, 768, 12, 2),
    (20, 128, 768, 12, 0),
    (1, 129, 64, 1, 3),        # few heads
    (3, 333, 320, 5, 3),
    (1, 1024, 768, 12, 3),
    (2, 1024, 1024, 8, 3),     # heads of 128
    (4, 333, 768, 12, 1),      # the forward's line lies above the backward's
    (8, 1024, 768, 12, 0),     # many heads: the kernels on 64- and 128-row blocks
    (4, 1024, 1600, 25, 0),
    (8, 333, 768, 12, 0),
    (10, 256, 1664, 13, 0),    # 130 heads of 128: a last round of workgroups that is nearly empty
    (1, 40, 6, 2, 0),          # head sizes that are no multiple of 4, or past 128
    (1, 40, 264, 2, 0),
])
def test_route(lib, B, T, C, H, route):
    assert lib.gptc_attention_slabs(B, T, C, H) == route


@pytest.mark.parametrize("D", [4, 48, 64, 96, 128])
@pytest.mark.parametrize("T", [130, 333, 1024, 2048])
def test_one_head_and_very_many(lib, D, T):
    assert lib.gptc_attention_slabs(1, T, D, 1) == 3
    assert lib.gptc_attention_slabs(1000, T, D, 1) == 0


def test_huge_rows_stay_off_the_slabs(lib):
    """A head's rows past 2^31 bytes (T x 3C floats) are outside a buffer's offsets."""
    assert lib.gptc_attention_slabs(1, 8000, 64 * 400, 400) == 0
    assert lib.gptc_attention_slabs(0, 128, 64, 1) == 0


def test_key_blocks_of_twenty_heads_are_cut(lib):
    """The shape that tests/test_attention_tiled_gpu.py takes for cut key blocks has some (2 workgroups a CU)."""
    import ctypes
    buf = [(ctypes.c_int * 20000)() for _ in range(2)]
    est, nsplit = ctypes.c_double(), ctypes.c_int()
    assert lib.gptc_attention_key_schedule(20, 16, 2, 32, buf[0], buf[1], 20000, ctypes.byref(est), ctypes.byref(nsplit)) > 0
    assert nsplit.value > 0
