"""The index arithmetic of the crowded passes' grouped kernels (launch_gsx, vitna-anchor_amd/csrc/kernels_tgemm.hip),
restated on the CPU. On random routings, and on routings that crowd every row onto the same K experts, at 64 to 1024 rows:
  * the plan: every pair in one tile slot, every tile in one token block of two (a fast pass: four), the blocks within the
    launch's grid and every (token block, row block) taken by one workgroup;
  * every load and store inside the buffer that the engine allocates (ensure_tiled);
  * the operands a lane reads from LDS are its token's columns, from what the image kernels wrote by way of the loads;
  * the LDS ring: what a step reads has landed and been waited for, and nothing is overwritten that a wave may still read.
The layout's numbers and the allocations are taken from the sources, so that neither can change without this.
"""
import os
import re

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vitna-anchor_amd", "csrc")
TGEMM = open(os.path.join(CSRC, "kernels_tgemm.hip")).read()
ENGINE = open(os.path.join(CSRC, "engine.hip")).read()

ROUTE_K_MAX, ROWS_MAX = 16, 1024
TG_R, TG_T = (int(re.search(r"#define %s (\d+)" % n, TGEMM).group(1)) for n in ("TG_R", "TG_T"))
THREADS, WAVES = 512, 8


class Lds:
    """tg_lds of one type."""

    def __init__(self, name):
        body = re.search(r"struct tg_lds<VITNA_DTYPE_%s> \{(.*?)\n\};" % name, TGEMM, re.S).group(1)
        self.name = name
        self.TB, self.WU, self.HDR_LANES = (int(re.search(r"\b%s = (\d+)" % n, body).group(1)) for n in ("TB", "WU", "HDR_LANES"))
        env = dict(TG_T=TG_T, TG_R=TG_R, WU=self.WU)
        for n in ("HDR", "QH", "SUMS", "BYTES"):
            m = re.search(r"int %s = ([^;]*);" % n, body)
            if m:
                env[n] = eval(m.group(1), {}, env)
                setattr(self, n, env[n])
        self.least = [eval(re.search(r"loads\(int u\) \{ return ([^;]*);", body).group(1), {}, dict(TG_T=TG_T, u=u)) for u in range(4)]
        self.slot = TG_T * 8192 + TG_R * self.WU


TYPES = {n: Lds(n) for n in ("Q4_K", "Q6_K", "Q8_0")}


def allocated(n_rows, K, E, H, I):
    """The buffers of ensure_tiled in bytes, from its own expressions."""
    T, W = max_tiles(n_rows, K, E), max(H, I)
    env = dict(T=T, W=W, H=H, I=I, E=E, ROWS_MAX=n_rows)
    out = {}
    for name, expr in re.findall(r"dalloc\(g, &g->gsx_(\w+), (.*?), \"scratch\"", ENGINE):
        out[name] = eval(expr.replace("g->", "").replace("sizeof(int)", "4").replace("/", "//"), {}, env)
    assert set(out) == {"toff", "te", "tb", "img_in", "img_act", "sums", "scale", "inv", "act"}
    return out


def max_tiles(n, K, E):
    return (n * K + 31) // 32 + E


def max_blocks(n, K, E):
    return (n * K + 63) // 64 + E


def plan(count, block):
    """gsx_plan_kernel: toff, te (-1 past the last), tb."""
    tiles, blocks = (count + 31) // 32, (count + 32 * block - 1) // (32 * block)
    toff = np.concatenate([[0], np.cumsum(tiles)])
    te = np.repeat(np.arange(len(count)), tiles)
    tb = np.concatenate([toff[e] + block * np.arange(blocks[e]) for e in range(len(count))])
    return toff, te, tb


def tiles_of(te, t, T, fast):
    """gsx_tiles: the tiles of the token block at t, and how many there are."""
    n = 1
    for j in range(1, 4 if fast else 2):
        n += n == j and t + j < T and te[t + j] == te[t]
    return n, [t + min(j, n - 1) for j in range(2 * TG_T)]


def item(block, n):
    """tg_item."""
    per, slot = (n + 7) >> 3, block >> 3
    w = (block & 7) * per + slot
    return w if slot < per and w < n else -1


def loads(dt, fast, S, tt, wv, b, U, part):
    """tg_part for wave wv: (source, source byte, LDS byte, bytes) of each load; sources img, wt (at the wave's tile), sums."""
    L = TYPES[dt]
    slot = U * L.slot
    if part < TG_T:
        if fast:
            src = tt[2 * part + (wv & 1)] * S * 16384 + (wv >> 1) * 1024 + b * 16384 + U * 4096
        else:
            src = tt[part] * S * 32768 + wv * 1024 + b * 32768 + U * 8192
        return [("img", src, slot + part * 8192 + wv * 1024, 1024)]
    out = [("wt", b * L.TB + U * L.WU + k * 1024, slot + TG_T * 8192 + wv * L.WU + k * 1024, 1024) for k in range(L.WU // 1024)]
    if dt == "Q6_K" and U % 2 == 0:
        out.append(("wt", b * L.TB + 4096 + U // 2 * 1024, L.QH + (U // 2 * TG_R + wv) * 1024, 1024))
    if U == 0:
        out.append(("wt", b * L.TB + 4 * L.WU + (2048 if dt == "Q6_K" else 0), L.HDR + wv * L.HDR_LANES * 16, L.HDR_LANES * 16))
        if dt == "Q4_K" and wv < 2 * TG_T:
            base = tt[wv & 3] * S * 2048 if fast else tt[(wv >> 1) & 1] * S * 2048 + (wv & 1) * 1024
            out.append(("sums", base + b * 2048, L.SUMS + wv * 1024, 1024))
    return out


def img_put(order, row, K, c8):
    """The 16-byte pieces (hi, lo) of columns 8 c8 .. of row `row` (skinny_image.h)."""
    b, c = c8 >> 5, 8 * (c8 & 31)
    base = ((row >> 5) * (K // 256) + b) * 2048
    if order == "a":
        U, r = c >> 6, c & 63
        i, kq = ((r >> 5) << 1) | ((r >> 3) & 1), (r >> 4) & 1
    else:
        r = c & 127
        U, i, kq = 2 * (c >> 7) + ((r >> 5) & 1), ((r >> 4) & 1) + 2 * (r >> 6), (r >> 3) & 1
    q = base + (U * 4 + i) * 2 * 64 + (row & 31) + 32 * kq
    return q, q + 64


def fast_put(order, row, K, c8):
    """gsx_put's piece of a fast pass."""
    order_b = order == "b"
    c = 8 * (c8 & 31)
    r = c & (127 if order_b else 63)
    U = 2 * (c >> 7) + ((r >> 5) & 1) if order_b else c >> 6
    kq = (r >> 3) & 1 if order_b else (r >> 4) & 1
    i = ((r >> 4) & 1) + 2 * (r >> 6) if order_b else ((r >> 5) << 1) | ((r >> 3) & 1)
    return ((row >> 5) * (K // 256) + (c8 >> 5)) * 1024 + (U * 4 + i) * 64 + (row & 31) + 32 * kq


def operand_c8(order, b, U, i, kq):
    """The first eighth column of operand i of unit U for lane half kq (skinny_image.h's two orders)."""
    if order == "a":
        return (256 * b + 64 * U + 16 * kq + 8 * (i % 2) + 32 * (i // 2)) // 8
    return (256 * b + 128 * (U // 2) + 32 * (U % 2) + 8 * kq + 16 * (i % 2) + 64 * (i // 2)) // 8


def check(n, K, E, H, I, ids, fast, gate_up="Q4_K", down="Q6_K"):
    T = max_tiles(n, K, E)
    have = allocated(ROWS_MAX, K, E, H, I)
    count = np.bincount(ids.ravel(), minlength=E)
    pairs = [[r * ROUTE_K_MAX + s for r in range(n) for s in range(K) if ids[r, s] == e] for e in range(E)]
    block = 4 if fast else 2
    toff, te, tb = plan(count, block)
    assert toff[-1] <= T and len(tb) <= max_blocks(n, K, E)
    assert 4 * (E + 1) <= have["toff"] and 4 * T <= have["te"] and 4 * n <= have["scale"]
    assert len(tb) <= max_tiles(ROWS_MAX, K, E) and 4 * (max_tiles(ROWS_MAX, K, E) + 1) <= have["tb"]
    # the plan's other blocks: every row's scale once
    assert sorted(4 * (b - 1) + w for b in range(1, 1 + (n + 3) // 4) for w in range(4) if 4 * (b - 1) + w < n) == list(range(n))
    te_full = np.concatenate([te, np.full(T - len(te), -1)])
    seen = np.zeros(toff[-1], int)
    for t in tb:
        m, tt = tiles_of(te_full, t, T, fast)
        assert (te_full[tt] == te_full[t]).all()
        seen[t:t + m] += 1
    assert (seen == 1).all(), "a tile in no token block, or in two"
    # the image kernels: rows read and written, and one pair a slot
    named = []
    for t in range(toff[-1]):
        e, j0 = te[t], 32 * (t - toff[te[t]])
        assert 0 <= j0 < count[e]
        for lane in range(32):
            assert pairs[e][min(j0 + lane, count[e] - 1)] // ROUTE_K_MAX < n
        named += [pairs[e][j] for j in range(j0, min(j0 + 32, count[e]))]
    assert sorted(named) == sorted(p for ps in pairs for p in ps)
    last = 32 * toff[-1] - 1
    for width, buf in ((H, "img_in"), (I, "img_act")):
        for order in "ab":
            most = max(fast_put(order, last, width, c8) if fast else max(img_put(order, last, width, c8)) for c8 in range(width // 8))
            assert 16 * (most + 1) <= have[buf]
        # th_sum: [tile][superblock][2][64][8] halves
        assert (((toff[-1] - 1) * (width // 256) + width // 256 - 1) * 1024 + 512 + (31 + 32) * 8 + 7 + 1) * 2 <= have["sums"]
    assert 4 * (last + 1) <= have["inv"] and 4 * (last + 1) * I <= have["act"]
    # the two kernels
    for dt, S, X, rows, img in ((gate_up, H // 256, I // 128, I, "img_in"), (down, I // 256, H // 256, H, "img_act")):
        L = TYPES[dt]
        grid = (max_blocks(n, K, E) * X + 7) // 8 * 8
        items = [item(b, len(tb) * X) for b in range(grid)]
        assert sorted(i for i in items if i >= 0) == list(range(len(tb) * X)), "a block's work left out or done twice"
        for it in {0, X - 1, len(tb) * X - 1, len(tb) * X // 2}:
            t, x = tb[it // X], it % X
            e = te[t]
            m, tt = tiles_of(te_full, t, T, fast)
            for wv in range(WAVES):
                tile = e * (rows // 32) + (4 * x + (wv >> 1) if img == "img_in" else TG_R * x + wv)
                assert tile < E * (rows // 32)
                for b in range(S):
                    for U in range(4):
                        for part in range(TG_T + 1):
                            for src, at, lds, size in loads(dt, fast, S, tt, wv, b, U, part):
                                limit = {"img": have[img], "sums": have["sums"], "wt": S * L.TB}[src]
                                assert 0 <= at and at + size <= limit, (src, at)
                                if src != "wt":  # this superblock of one of the block's tiles
                                    per = 2048 if src == "sums" else 16384 if fast else 32768
                                    assert at // (S * per) in tt and at // per % S == b and (at + size - 1) // per == at // per
                                assert lds % 16 == 0 and lds + size <= L.BYTES
        assert L.BYTES <= 160 * 1024
    # the results: gate/up's rows of the tiles that there are, down's pairs
    assert 32 * (4 * (I // 128 - 1) + 3) + 31 < I and 32 * (TG_R * (H // 256 - 1) + 2 * 3) + 31 + 32 < H
    assert max(p // ROUTE_K_MAX for p in named) < n and max(p % ROUTE_K_MAX for p in named) < K


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("n,K,E,H,I", [(64, 8, 128, 2048, 768), (1024, 8, 128, 2048, 768), (520, 8, 32, 512, 256),
                                       (600, 4, 16, 256, 256), (1024, 4, 16, 512, 256), (333, 8, 64, 2048, 1024), (72, 2, 8, 2048, 2048)])
def test_random_routing(n, K, E, H, I, fast):
    rng = np.random.default_rng(n * 7 + E)
    ids = np.stack([np.sort(rng.choice(E, K, replace=False)) for _ in range(n)])
    check(n, K, E, H, I, ids, fast)
    check(n, K, E, H, I, ids, fast, "Q6_K", "Q4_K")
    if not fast:
        check(n, K, E, H, I, ids, fast, "Q8_0", "Q8_0")


@pytest.mark.parametrize("n", [64, 65, 333, 1024])
def test_crowded_routing(n):
    """Every row on the same K experts: each of them holds n pairs (n / 32 tiles, the last part-filled)."""
    K, E = 8, 128
    ids = np.tile(np.arange(3, 3 + K), (n, 1))
    for fast in (False, True):
        check(n, K, E, 2048, 768, ids, fast)


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("dt", ["Q4_K", "Q6_K", "Q8_0"])
def test_operands_of_a_lane(dt, fast):
    """Images of five tiles written piece by piece, brought to LDS by the eight waves' loads, read back as tg_read_a does."""
    if fast and dt == "Q8_0":
        return
    K, S, tiles, order = 512, 2, 5, "b" if dt == "Q6_K" else "a"
    img = {}
    for row in range(32 * tiles):
        for c8 in range(K // 8):
            if fast:
                assert img.setdefault(fast_put(order, row, K, c8), (row, c8, 0)) == (row, c8, 0)
            else:
                for hl, q in enumerate(img_put(order, row, K, c8)):
                    assert img.setdefault(q, (row, c8, hl)) == (row, c8, hl)
    assert sorted(img) == list(range(tiles * S * (1024 if fast else 2048)))
    tt = [1, 2, 3, 4] if fast else [3, 1, 1, 1]
    L = TYPES[dt]
    for b in range(S):
        for U in range(4):
            lds = {}
            for wv in range(WAVES):
                for part in range(TG_T):
                    for _, at, to, size in loads(dt, fast, S, tt, wv, b, U, part):
                        for lane in range(size // 16):
                            assert to // 16 + lane not in lds
                            lds[to // 16 + lane] = img[at // 16 + lane]
            for tg in range(2):
                for lane in range(64):
                    p = (U * L.slot + tg * 8192) // 16 + lane
                    for i in range(4):
                        c8 = operand_c8(order, b, U, i, lane >> 5)
                        h, lo = lds[p + i * 128], lds[p + i * 128 + 64]
                        if fast:
                            assert h == (32 * tt[2 * tg] + lane % 32, c8, 0) and lo == (32 * tt[2 * tg + 1] + lane % 32, c8, 0)
                        else:
                            assert h == (32 * tt[tg] + lane % 32, c8, 0) and lo == (32 * tt[tg] + lane % 32, c8, 1)


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("dt", ["Q4_K", "Q6_K", "Q8_0"])
@pytest.mark.parametrize("S", [1, 2, 3, 8])
def test_ring(dt, fast, S):
    """tg_body's order of loads, waits and reads. A wait and barrier begins a segment: what a wave reads in one was landed
    for every wave by its wait, and what it loads into is not read by any wave in the same one."""
    if fast and dt == "Q8_0":
        return
    L = TYPES[dt]
    tt = [0, 1, 2, 3] if fast else [0, 1, 1, 1]

    def regions(U):
        """What a step may read of unit U: name -> LDS bytes of all waves' loads."""
        r = {}
        for wv in range(WAVES):
            for part in range(TG_T + 1):
                for src, _, to, size in loads(dt, fast, S, tt, wv, 0, U, part):
                    where = "slot" if to < L.HDR else "sums" if src == "sums" else "qh" if dt == "Q6_K" and L.QH <= to else "hdr"
                    r.setdefault(where, []).append((to, to + size))
        return r

    # what lies where never overlaps: the four slots, the headers, the high bits, the sums
    spans = sorted(s for U in range(4) for rs in regions(U).values() for s in rs)
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])) and spans[-1][1] <= L.BYTES
    for wv in range(WAVES):
        issued, segments = [], []  # loads (region, b) of this wave; each segment's waited loads, loads and reads

        def issue(U, b):
            for part in range(TG_T + 1):
                for src, _, to, _ in loads(dt, fast, S, tt, wv, b, U, part):
                    where = ("slot", U) if to < L.HDR else ("sums",) if src == "sums" else ("qh", U // 2) if dt == "Q6_K" and L.QH <= to else ("hdr",)
                    issued.append((where, b))
                    if segments:
                        segments[-1]["loads"].append((where, b))

        def wait(n):
            segments.append(dict(landed=set(issued[:len(issued) - n] if n else issued), loads=[], reads=[]))

        def read(*what):
            segments[-1]["reads"].append(what)

        def weights(U, b):
            read(("slot", U), b)
            if dt == "Q6_K" and U % 2 == 0:
                read(("qh", U // 2), b)
            if U == 0:
                read(("hdr",), b)

        for U in range(3):
            issue(U, 0)
            assert len([1 for p in range(TG_T + 1) for _ in loads(dt, fast, S, tt, wv, 0, U, p)]) >= L.least[U]
        wait(L.least[1] + L.least[2])
        weights(0, 0)
        if dt == "Q4_K" and wv < 2 * TG_T:
            read(("sums",), 0)
        for b in range(S):
            for U in range(4):
                V = (U + 1) & 3
                wait(L.least[(U + 2) & 3] if U < 2 or b + 1 < S else 0)
                if U == 0:
                    issue(3, b)
                elif b + 1 < S:
                    issue((U + 3) & 3, b + 1)
                read(("slot", U), b)
                if U < 3 or b + 1 < S:  # past the last superblock what is read is not used
                    weights(V, b + (U == 3))
                    if dt == "Q4_K" and U == 3 and wv < 2 * TG_T:
                        read(("sums",), b + 1)
        assert segments[-1]["landed"] == set(issued), "loads under way at the kernel's end"
        current = {}
        for s in segments:
            for where, b in s["reads"]:
                assert (where, b) in s["landed"], (where, b)
                assert current.get(where, b) <= b
                current[where] = b
            busy = {w for w, _ in s["reads"]}
            for where, b in s["loads"]:
                assert where not in busy, ("overwritten while it is read", where, b)
                # the version before it has been read for the last time
                assert all((where, b - 1) not in later["reads"] for later in segments[segments.index(s):]), (where, b)
