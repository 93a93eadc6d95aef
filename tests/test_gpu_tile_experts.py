"""The grouped experts of crowded passes at the edges of their tiles: 32 pairs a tile, two tiles a block, 256 weight
rows a block, whole superblocks of the width. The caller's routing (vitna_cuda_moe_rows_experts takes any) puts 1, 31,
32, 33, 63, 64, 65, 96, 97 and 129 pairs on the experts of one layer and none on others, for every pair of types, one
superblock and several, and scales at which the SwiGLU output leaves float16's range on either side.

The oracle: each row's mixture from the checker's norm, projections and SwiGLU on the device's residual rows, to the
grouped experts' bar of 1e-4 of max |mixture| (float32 sums in another order).
"""
import numpy as np
import pytest

import oracle
import vitna_amd as va
from test_gpu_decode import say

pytestmark = pytest.mark.gpu

REL = 1e-4
COUNTS = [1, 31, 32, 33, 63, 64, 65, 96, 97, 129]


def routing(n, E, K, seed):
    """ids n x K (ascending, distinct): expert i takes COUNTS[i] pairs, the remaining pairs go to the experts after."""
    rng = np.random.RandomState(seed)
    left = {e: c for e, c in enumerate(COUNTS)}
    ids = [[] for _ in range(n)]
    for e, c in left.items():
        for r in rng.permutation([r for r in range(n) if len(ids[r]) < K])[:c]:
            ids[r].append(e)
    rest = list(range(len(COUNTS), E - 1))  # the last expert takes none
    for r in range(n):
        while len(ids[r]) < K:
            e = rest[rng.randint(len(rest))]
            if e not in ids[r]:
                ids[r].append(e)
    ids = np.sort(np.array(ids, np.int32), axis=1)
    w = rng.uniform(0.05, 1.0, (n, K)).astype(np.float32)
    return ids, w


def mixture(model, layer, xn, ids, w):
    experts = model.m.layers[layer].experts
    out = np.zeros(model.cfg.hidden, np.float32)
    for e, wt in zip(ids, w):
        x = experts[int(e)]
        mv = lambda m, v: oracle.matvec(m.data, m.dtype, v, m.rows, m.cols)
        out = out + mv(x.down, oracle.silu_mul(mv(x.gate, xn), mv(x.up, xn))) * wt
    return out


@pytest.mark.parametrize("gate_up,down", [(va.Q4_K, va.Q6_K), (va.Q6_K, va.Q4_K), (va.Q4_K, va.Q4_K), (va.Q6_K, va.Q6_K), (va.Q8_0, va.Q8_0)])
@pytest.mark.parametrize("hidden,inter,k_scale,q8_scale", [(256, 256, 0.01, 0.02 / 127), (512, 768, 3.0, 40.0 / 127), (1024, 256, 2e-4, 5e-3 / 127)])
def test_tile_edges(gate_up, down, hidden, inter, k_scale, q8_scale):
    say("tile edges", gate_up, down, hidden, inter, k_scale)
    n, E, K = 200, 24, 4
    model = va.Model(va.shape(n_layers=1, hidden=hidden, intermediate=inter, n_heads=4, n_kv_heads=2, head_dim=64, vocab=300, n_experts=E,
                              n_experts_used=K, renormalize=0, dt_gate_up=gate_up, dt_down=down, norm_std=0.5, k_scale=k_scale,
                              q8_scale=q8_scale, ctx=n + 8, seqs=1), 977)
    dev = va.Device(model)
    try:
        cfg = model.cfg
        rows = [((11 * i + 7) % cfg.vocab, i, 0) for i in range(n)]
        dev.rows_route(rows, 0)
        norm = np.ctypeslib.as_array(model.m.layers[0].mlp_norm, shape=(hidden,)).copy()
        x0 = np.stack([dev.residual(i) for i in range(n)])
        ids, w = routing(n, E, K, 5)
        dev.rows_experts(0, ids, w)
        x1 = np.stack([dev.residual(i) for i in range(n)])
        worst = 0.0
        for i in range(n):
            ref = mixture(model, 0, oracle.rmsnorm(x0[i], norm, cfg.rms_eps), ids[i], w[i])
            want = x0[i].astype(np.float64) + ref
            r = float(np.max(np.abs(x1[i] - want)) / np.max(np.abs(ref)))
            # what float32 keeps of a small mixture beside its residual
            lost = float(np.max(np.abs(want))) * 2.0 ** -23 / float(np.max(np.abs(ref)))
            worst = max(worst, r)
            assert r <= REL + lost, ("row", i, r, lost)
        say("  worst rel err of the mixture", worst)
    finally:
        dev.close()
        model.free()


def fast_bound(model, layer, xn, ids, w):
    """A fast pass's mixture and its bound: activations, weights and SwiGLU outputs each within 2^-11 of themselves (f16), so
    a product within 2^-10; the gate's and up's error carried through SwiGLU to first order, and 5 % for the rest."""
    e10 = 2.0 ** -10
    out, bound = np.zeros(model.cfg.hidden), np.zeros(model.cfg.hidden)
    for e, wt in zip(ids, w):
        x = model.m.layers[layer].experts[int(e)]
        G, U, D = (oracle.widen(m.bytes(), m.dtype, m.rows * m.cols).reshape(m.rows, m.cols).astype(np.float64) for m in (x.gate, x.up, x.down))
        xd = xn.astype(np.float64)
        g, u = G @ xd, U @ xd
        dg, du = e10 * (np.abs(G) @ np.abs(xd)), e10 * (np.abs(U) @ np.abs(xd))
        sg = 1.0 / (1.0 + np.exp(-np.clip(g, -700, 700)))
        a = g * sg * u
        # |silu'| is at most 1.1 everywhere
        da = 1.1 * np.abs(u) * dg + (np.abs(g * sg) + 1.1 * dg) * du
        out += wt * (D @ a)
        bound += abs(wt) * (np.abs(D) @ (da + e10 * np.abs(a)))
    return out, 1.05 * bound


@pytest.mark.parametrize("gate_up,down", [(va.Q4_K, va.Q6_K), (va.Q6_K, va.Q4_K)])
@pytest.mark.parametrize("hidden,inter", [(256, 256), (512, 768)])
def test_fast_tile_edges(gate_up, down, hidden, inter):
    """The same pairs an expert through a --precision fast model: blocks of four tiles of one expert."""
    say("fast tile edges", gate_up, down, hidden, inter)
    n, E, K = 200, 24, 4
    model = va.Model(va.shape(n_layers=1, hidden=hidden, intermediate=inter, n_heads=4, n_kv_heads=2, head_dim=64, vocab=300, n_experts=E,
                              n_experts_used=K, renormalize=0, dt_gate_up=gate_up, dt_down=down, norm_std=0.5, ctx=n + 8, seqs=1), 978)
    dev = va.Device(model, fast=True)
    try:
        cfg = model.cfg
        rows = [((11 * i + 7) % cfg.vocab, i, 0) for i in range(n)]
        dev.rows_route(rows, 0)
        norm = np.ctypeslib.as_array(model.m.layers[0].mlp_norm, shape=(hidden,)).copy()
        x0 = np.stack([dev.residual(i) for i in range(n)])
        ids, w = routing(n, E, K, 6)
        dev.rows_experts(0, ids, w)
        worst = 0.0
        for i in range(0, n, 3):
            ref, bound = fast_bound(model, 0, oracle.rmsnorm(x0[i], norm, cfg.rms_eps), ids[i], w[i])
            got = dev.residual(i).astype(np.float64) - x0[i]
            r = float(np.max(np.abs(got - ref) / bound))
            worst = max(worst, r)
            assert r <= 1.0, ("row", i, r)
        say("  worst share of the bound", worst)
    finally:
        dev.close()
        model.free()


def given_rows(model, dev, n):
    """A pass of n rows of one sequence up to its experts: their residual rows and normalized rows."""
    cfg = model.cfg
    dev.rows_route([((11 * i + 7) % cfg.vocab, i, 0) for i in range(n)], 0)
    norm = np.ctypeslib.as_array(model.m.layers[0].mlp_norm, shape=(cfg.hidden,)).copy()
    x0 = np.stack([dev.residual(i) for i in range(n)])
    return x0, np.stack([oracle.rmsnorm(x, norm, cfg.rms_eps) for x in x0])


def check_mixture(model, dev, ids, w, bar):
    """The mixture of given rows against the oracle's, to bar and what float32 keeps of it beside its residual row."""
    n = len(ids)
    x0, xn = given_rows(model, dev, n)
    dev.rows_experts(0, ids, w)
    worst = 0.0
    for i in range(n):
        ref = mixture(model, 0, xn[i], ids[i], w[i]).astype(np.float64)
        got = dev.residual(i).astype(np.float64) - x0[i]
        assert np.isfinite(ref).all() and np.isfinite(got).all(), ("row", i)
        most = float(np.max(np.abs(ref)))
        lost = float(np.max(np.abs(x0[i].astype(np.float64) + ref))) * 2.0 ** -23 / most
        r = float(np.max(np.abs(got - ref)) / most)
        worst = max(worst, r)
        assert r <= bar + lost, ("row", i, r, lost)
    say("  worst rel err of the mixture", worst)


@pytest.mark.parametrize("gate_up,down,scale", [(va.Q8_0, va.Q6_K, 2.0 ** 62), (va.Q4_K, va.Q8_0, 2.0 ** 59), (va.Q6_K, va.Q8_0, 2.0 ** 60)])
def test_large_activations(gate_up, down, scale):
    """Norm weights of 2^60: normalized rows of that size and SwiGLU outputs above 2^116, which the f16 operands hold by the
    row's own power of two; the mixture is finite, as in float32."""
    say("large activations", gate_up, down)
    model = va.Model(va.shape(n_layers=1, hidden=256, intermediate=256, n_heads=4, n_kv_heads=2, head_dim=64, vocab=300, n_experts=24,
                              n_experts_used=4, renormalize=0, dt_gate_up=gate_up, dt_down=down, norm_std=0.5, k_scale=1e-4,
                              q8_scale=0.02 / 127, ctx=208, seqs=1), 980)
    norm = np.ctypeslib.as_array(model.m.layers[0].mlp_norm, shape=(256,))
    norm *= np.float32(scale)
    dev = va.Device(model)
    try:
        check_mixture(model, dev, *routing(200, 24, 4, 7), REL)
    finally:
        dev.close()
        model.free()


def all_of(dtype):
    return {"dt_" + m: dtype for m in ("q", "k", "v", "o", "embed")}


@pytest.mark.parametrize("gate_up,down,k_scale,q8_scale,eps", [(va.Q8_0, va.Q6_K, 1e-4, 10000.0, 2.0 ** 48), (va.Q4_K, va.Q8_0, 10000.0, 1e-3, 2.0 ** 60),
                                                               (va.Q6_K, va.Q8_0, 3000.0, 1e-3, 2.0 ** 54)])
def test_rows_far_below_their_bound(gate_up, down, k_scale, q8_scale, eps):
    """An epsilon that makes normalized rows some 2^-30 of the largest that the norm's weights allow: a row's operands hold
    it as well as any other's, so its mixture is within the same bar."""
    say("rows far below their bound", gate_up, down)
    model = va.Model(va.shape(n_layers=1, hidden=256, intermediate=256, n_heads=4, n_kv_heads=2, head_dim=64, vocab=300, n_experts=24,
                              n_experts_used=4, renormalize=0, dt_gate_up=gate_up, dt_down=down, norm_std=0.5, k_scale=k_scale,
                              q8_scale=q8_scale, rms_eps=eps, ctx=208, seqs=1, **all_of(va.Q4_K if gate_up == va.Q8_0 else va.Q8_0)), 980)
    dev = va.Device(model)
    try:
        check_mixture(model, dev, *routing(200, 24, 4, 8), REL)
    finally:
        dev.close()
        model.free()


@pytest.mark.parametrize("experts,gate_up,down", [(16, va.Q4_K, va.Q6_K), (16, va.Q6_K, va.Q4_K), (16, va.Q8_0, va.Q8_0), (40, va.Q4_K, va.Q6_K),
                                                  (40, va.Q8_0, va.Q4_K)])
@pytest.mark.parametrize("n", [63, 64, 71, 72, 95, 96])
def test_first_tiled_passes(experts, gate_up, down, n):
    """Passes about the first ones on the tiles: 64 rows, and 96 for K-quant experts with few blocks (16 experts of 512 x 256
    have 32, 40 have 80), the kernels on either side of the limit to the grouped experts' bar."""
    say("first tiled passes", experts, gate_up, down, n)
    model = va.Model(va.shape(n_layers=1, hidden=512, intermediate=256, n_heads=4, n_kv_heads=2, head_dim=64, vocab=300, n_experts=experts,
                              n_experts_used=4, renormalize=0, dt_gate_up=gate_up, dt_down=down, norm_std=0.5, ctx=n, seqs=1), 981)
    dev = va.Device(model)
    try:
        dev.set_exact_rows(0)
        rng = np.random.RandomState(n)
        ids = np.stack([np.sort(rng.choice(experts, 4, replace=False)) for _ in range(n)]).astype(np.int32)
        check_mixture(model, dev, ids, rng.uniform(0.05, 1.0, (n, 4)).astype(np.float32), REL)
    finally:
        dev.close()
        model.free()


@pytest.mark.parametrize("gate_up,down,fast", [(a, b, f) for a, b in ((va.Q4_K, va.Q4_K), (va.Q6_K, va.Q6_K), (va.Q4_K, va.Q6_K))
                                               for f in (False, True)] + [(va.Q8_0, va.Q8_0, False)])
def test_widest_experts(gate_up, down, fast):
    """Experts of 2048 x 2048, the widest on the tiles (a fast pass's Q8_0 ones keep the prefill's kernel): some of 97 rows,
    two experts each, to the bars above."""
    say("widest experts", gate_up, down, fast)
    n, E, K = 97, 8, 2
    model = va.Model(va.shape(n_layers=1, hidden=2048, intermediate=2048, n_heads=4, n_kv_heads=2, head_dim=64, vocab=300, n_experts=E,
                              n_experts_used=K, renormalize=0, dt_gate_up=gate_up, dt_down=down, norm_std=0.5, ctx=n, seqs=1), 982)
    dev = va.Device(model, fast=fast)
    try:
        x0, xn = given_rows(model, dev, n)
        rng = np.random.RandomState(4)
        ids = np.stack([np.sort(rng.choice(E - 1, K, replace=False)) for _ in range(n)]).astype(np.int32)
        w = rng.uniform(0.05, 1.0, (n, K)).astype(np.float32)
        dev.rows_experts(0, ids, w)
        for i in range(0, n, 12):
            ref, bound = fast_bound(model, 0, xn[i], ids[i], w[i])
            got = dev.residual(i).astype(np.float64) - x0[i]
            most = float(np.max(np.abs(ref)))
            lost = float(np.max(np.abs(x0[i] + ref))) * 2.0 ** -23
            assert np.max(np.abs(got - ref) / (bound + lost) if fast else np.abs(got - ref) / (REL * most + lost)) <= 1.0, ("row", i)
    finally:
        dev.close()
        model.free()
