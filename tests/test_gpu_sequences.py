"""How the engine tells a pass's sequences apart. A model without attention has no cache, and any number of sequences in
its description costs nothing; rows of sequences that meet in one slot of the pass's table are told apart, and two rows
of one sequence are seen wherever they stand.
"""
import numpy as np
import pytest

import vitna_amd as va
from test_gpu_decode import say
from test_gpu_exact_rows import as_pass, check, one_at_a_time

pytestmark = pytest.mark.gpu


def small(**more):
    spec = dict(n_layers=1, hidden=512, intermediate=256, n_experts=16, n_experts_used=4, norm_std=0.1, ctx=16, seqs=1)
    return va.Model(va.shape(**dict(spec, **more)), 1357)


def test_sequences_of_a_model_without_attention():
    say("no attention", "2^61 sequences")
    x = va.normal(5, 1, 7 * 512).reshape(7, 512)
    model = small(attention=0)
    try:
        got = []
        for seqs in (1, 1 << 61):
            model.m.seqs = seqs
            dev = va.Device(model)
            try:
                got.append(dev.prefill(0, x))
            finally:
                dev.close()
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    finally:
        model.m.seqs = 1
        model.free()


def test_sequences_that_meet_in_a_slot():
    say("sequences", 0, 2048, 1)
    a, b, c = 0, 2048, 1  # b's slot is a's, so it takes c's
    model = small(n_heads=4, n_kv_heads=2, head_dim=128, vocab=1000, seqs=2049)
    # each sequence's later rows need the keys of its earlier ones
    passes = [[(3, 0, a), (5, 0, b), (8, 0, c)], [(7, 1, a), (9, 1, b), (11, 1, c), (13, 2, b)],
              [(2, 3, b), (4, 2, c), (6, 2, a), (8, 3, a), (1, 3, c)]]
    dev, one = va.Device(model), va.Device(model)
    try:
        for rows in passes:
            check(model.cfg, rows, one_at_a_time(one, model.cfg, rows), as_pass(dev, model.cfg, rows), one, dev)
    finally:
        dev.close()
        one.close()
        model.free()
