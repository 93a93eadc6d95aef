"""Results copied to the host through page-locked chunks of 512 KB (csrc/host_copy.hip): the bytes against the same
results read by other calls, at the edges of a chunk, of the plain copies' range (64 KB to 2 MB) and of the ring of
chunks (16 MB)."""

import numpy as np
import pytest

import vitna_amd as va
from test_gpu_decode import say

pytestmark = pytest.mark.gpu

HIDDEN = 1024
SPEC = dict(n_layers=1, hidden=HIDDEN, intermediate=256, n_heads=8, n_kv_heads=2, head_dim=128, vocab=32771, n_experts=8,
            n_experts_used=2, norm_std=0.1, ctx=64, kv_host=1, seqs=40)


@pytest.fixture(scope="module")
def dev():
    model = va.Model(va.shape(**SPEC), 4242)
    d = va.Device(model)
    yield d
    d.close()
    model.free()


@pytest.mark.parametrize("n", [1, 16, 17, 128, 511, 512, 513, 4095, 4096, 4097, 9000])
def test_prefilled_rows(dev, n):
    """n rows of 4 KB: into a new array and in place, against the device's rows read with one plain copy."""
    say("prefilled rows", n)
    x = np.random.RandomState(n).standard_normal((n, HIDDEN)).astype(np.float32)
    kept = x.copy()
    out, chosen = dev.prefill(0, x)
    assert np.array_equal(x, kept)
    first, rows, ids = dev.prefill_rows(n)
    assert np.array_equal(out.view(np.uint32), rows.view(np.uint32)) and np.array_equal(chosen, ids)
    dev._ok(dev.lib.vitna_hip_moe_prefill(dev.g, 0, va.fptr(x), n, None, dev.err, 512))
    assert np.array_equal(x.view(np.uint32), out.view(np.uint32))


@pytest.mark.parametrize("only", [None, [], [0], [39], [0, 1, 2, 5, 17, 18, 19, 39], range(3, 39)])
def test_rows_of_logits(dev, only):
    """40 rows of 131084 bytes (chunks end inside rows), all, none, single ones and runs of them, in chunks and in
    plain copies: each as in the pass that copies all, the others' memory untouched."""
    rows = [(7 * i, 0, i) for i in range(40)]
    every = dev.rows_step(rows)
    out = np.full_like(every, 7.0)
    dev._ok(dev.lib.vitna_hip_moe_rows_step(dev.g, dev._rows(rows), 40, dev._row_pointers(out, only), dev.err, 512))
    want = set(range(40) if only is None else only)
    for i in range(40):
        assert np.array_equal(out[i], every[i]) if i in want else (out[i] == 7.0).all(), i
