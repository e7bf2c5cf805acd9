"""The one-token step at the edges of its row kernels (csrc/decode_ops.hip): 1 to 8
sequences (one row, and 2, 4 and 8 rows held), widths that fill their 16-byte
vectors partly, the widest that a wave holds and one past it; each against the
model's forward over the sequence, within the 1e-4 x the largest logit of the
other decode tests."""
import numpy as np
import pytest

import gptc
from test_generate_gpu import c3_params, check, make_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,C", [
    (1, 6, 384), (2, 6, 384), (3, 6, 384), (4, 6, 384), (5, 6, 384), (8, 6, 384),
    (1, 4, 260), (7, 4, 260),    # 65 vectors a row
    (1, 16, 1024), (6, 16, 1024), (2, 16, 1024),
    (1, 13, 1040), (8, 13, 1040),
    (4, 3, 342), (1, 3, 342), (2, 3, 342), (7, 3, 342), (1, 3, 771), (3, 3, 771),  # rows that are no whole vectors
])
def test_decode_rows(rt, B, H, C):
    print(f"case decode rows B={B} H={H} C={C}", flush=True)
    V, block, T = 53, 8, 4
    model = make_model(rt, c3_params(V, block, 2, C, seed=B + C, std=0.05, jitter=0.05), V, block, 2, H, C)
    seq = np.random.default_rng(C).integers(0, V, (B, T))
    cache = gptc.KVCache(rt, model, B, T)
    dec = np.empty((B, T, V), np.float32)
    for pos in range(T):
        ids = rt.from_numpy(seq[:, pos:pos + 1].astype(np.float32))
        lt = cache.decode(ids, pos)
        dec[:, pos] = rt.to_numpy(lt)[:, 0]
        rt.free(lt)
        rt.free(ids)
    cache.free()
    lt = model.forward(rt.from_numpy(seq.astype(np.float32)))
    fwd = rt.to_numpy(lt)
    rt.free(lt)
    model.free_cache()
    model.free()
    check("decode vs forward", dec, fwd)
