"""The rows step's captured graphs: a pass of one sequence (attention over tiles of its rows) and a pass of as many rows
of two sequences have graphs of their own, also where everything else of the two passes is alike (rows, attention
grid, the head's rows). Each pass in turn on one device, bit for bit the logits and attention outputs of the same
passes on devices that never ran the other kind.
"""
import numpy as np
import pytest

import vitna_amd as va
from test_gpu_decode import say

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("heads,kvs,start,n", [(4, 2, 40, 4), (8, 2, 300, 12), (8, 1, 400, 80)])
def test_one_sequence_and_two_in_turn(heads, kvs, start, n):
    say("rows graphs", heads, kvs, "rows", start, n)
    model = va.Model(va.shape(n_layers=1, hidden=512, intermediate=256, n_heads=heads, n_kv_heads=kvs, head_dim=128, vocab=1000,
                              n_experts=16, n_experts_used=4, norm_std=0.1, ctx=start + n, seqs=2), 8642)
    kd = kvs * 128
    one = [((13 * i + 5) % 1000, start + i, 0) for i in range(n)]
    # the first rows the same, the second half another sequence's; the last position too, for the same grid
    two = one[:n // 2] + [((17 * i + 3) % 1000, start + i, 1) for i in range(n // 2, n)]

    def fresh():
        dev = va.Device(model)
        for seq in range(2):
            dev.kv(seq, 0, 0, start + n, va.normal(3, 2 * seq + 1, (start + n) * kd).reshape(-1, kd),
                   va.normal(3, 2 * seq + 2, (start + n) * kd).reshape(-1, kd))
        return dev

    def run(dev, rows):
        logits = dev.rows_step(rows)
        return bits(logits), bits(np.stack([dev.attention_io(i)[1] for i in range(n)]))

    a, b, both = fresh(), fresh(), fresh()
    try:
        want = {"one": run(a, one), "two": run(b, two)}
        for turn, (kind, rows) in enumerate([("one", one), ("two", two), ("one", one), ("two", two)]):
            logits, att = run(both, rows)
            assert np.array_equal(att, want[kind][1]), (turn, kind, "attention rows", np.nonzero((att != want[kind][1]).any(1))[0])
            assert np.array_equal(logits, want[kind][0]), (turn, kind)
    finally:
        for dev in (a, b, both):
            dev.close()
        model.free()
