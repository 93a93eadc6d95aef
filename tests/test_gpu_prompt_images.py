"""A prompt pass's attention from the chunks' images (eight row tiles or more) against the same rows in passes of fewer
tiles, whose blocks split the chunks themselves: the same bits of every row's attention output, for passes that start
before, on and after a 64-position chunk's edge, with a last tile part-filled, at 8, 4, 2 and 1 query heads a kv head, and
for rows out of the order of their positions.
One layer, so that the rows' queries, keys and values are the same bits however the pass is cut.
"""
import numpy as np
import pytest

import vitna_amd as va
from test_gpu_decode import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kvs", [(16, 2), (8, 2), (4, 2), (2, 2)])
@pytest.mark.parametrize("start,n", [(0, 520), (63, 513), (64, 577), (190, 600)])
def test_images_against_own_split(heads, kvs, start, n):
    say("prompt images", heads, kvs, "rows", start, n)
    model = va.Model(va.shape(n_layers=1, hidden=512, intermediate=256, n_heads=heads, n_kv_heads=kvs, head_dim=128, vocab=1000, n_experts=16,
                              n_experts_used=4, norm_std=0.1, ctx=start + n, seqs=1), 1357)
    a, b = va.Device(model), va.Device(model)
    try:
        kd = kvs * 128
        k, v = va.normal(3, 1, start * kd + 1)[:start * kd].reshape(start, kd), va.normal(3, 2, start * kd + 1)[:start * kd].reshape(start, kd)
        for d in (a, b):
            if start:
                d.kv(0, 0, 0, start, k, v)
        rows = [((13 * i + 5) % 1000, start + i, 0) for i in range(n)]
        a.rows_step(rows, logits=False)
        piece = 7 * 4 * (16 // (heads // kvs))  # seven tiles
        for at in range(0, n, piece):
            some = rows[at:at + piece]
            b.rows_step(some, logits=False)
            if len(some) == 1:
                continue  # a single row takes the decode kernels
            for i in range(0, len(some), 5):
                got, want = a.attention_io(at + i)[1], b.attention_io(i)[1]
                assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), ("row", at + i)
    finally:
        a.close()
        b.close()
        model.free()


@pytest.mark.parametrize("n", [72, 200])
def test_rows_out_of_order(n):
    """Rows whose positions run backwards, every second one first: each tile's last position is another than its last row's.
    Against the same rows in their order on a device of its own."""
    say("prompt images, rows out of order", n)
    start = 400
    model = va.Model(va.shape(n_layers=1, hidden=512, intermediate=256, n_heads=16, n_kv_heads=2, head_dim=128, vocab=1000, n_experts=16,
                              n_experts_used=4, norm_std=0.1, ctx=start + n, seqs=1), 1357)
    a, b = va.Device(model), va.Device(model)
    try:
        k, v = va.normal(3, 1, start * 256).reshape(start, 256), va.normal(3, 2, start * 256).reshape(start, 256)
        rows = [((13 * i + 5) % 1000, start + i, 0) for i in range(n)]
        order = list(range(n - 1, -1, -2)) + list(range(n - 2, -1, -2))
        for d, some in ((a, [rows[i] for i in order]), (b, rows)):
            d.kv(0, 0, 0, start, k, v)
            d.rows_step(some, logits=False)
        for at, i in enumerate(order):
            got, want = a.attention_io(at)[1].astype(np.float64), b.attention_io(i)[1].astype(np.float64)
            # a row's chunks are summed in one order whatever its tile; only the split of the products differs by tile
            assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want)), ("row", i)
    finally:
        a.close()
        b.close()
        model.free()
