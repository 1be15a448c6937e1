"""CPU model of the prefill kernel's equal ranges (csrc/varlen_prefill.hip,
``Ranges``): for ragged batches, every live item's key tiles are covered
exactly once, a cut falls on a cache-block boundary, each range holds at most
one continued and one continuing item, and the merge's walk from an item's
first piece meets exactly its other pieces."""
import ctypes
import random

import pytest
import torch

from nano_qwen_amd._lib import dtype_code, lib

KEYS, ITEM, MIN = 32, 8, 2


def cdiv(a, b):
    return -(-a // b)


class Queue:
    """One XCD's queue: entries (sequence, own query tile, slot) and costs."""

    def __init__(self, x, lq, lk, n_y, rows, pin, rep, n_wg, tpb, causal):
        n_x = max(cdiv(q, rows) for q in lq)
        r = x // n_y if rep > 1 else 0
        self.n_own = (n_x + rep - 1 - r) // rep if n_x > r else 0
        self.w = 1 if rep > 1 else (cdiv(n_y, 8) if pin else n_y)
        self.gran = tpb if tpb >= 4 else tpb * ((3 + tpb) // tpb)
        self.tpb, self.n_wg = tpb, n_wg
        self.items, self.cum = [], [0]
        for s in range(len(lq)):
            y0 = x % n_y if rep > 1 else ((x - s * n_y) % 8 if pin else 0)
            for k in range(self.n_own):
                for yi in range(self.w):
                    y, qt = y0 + (8 if pin else 1) * yi, k * rep + r
                    live = y < n_y and qt * rows < lq[s]
                    end = (max(0, min(lk[s], min((qt + 1) * rows, lq[s]) + lk[s] - lq[s])) if causal else lk[s])
                    self.items.append((s, y, qt, cdiv(end, KEYS)) if live else None)
                    self.cum.append(self.cum[-1] + (cdiv(end, KEYS) + ITEM if live else 0))
        total = self.cum[-1]
        self.n_rg = max(1, min(n_wg, total // (2 * MIN + ITEM)))
        self.bounds = [w * total // self.n_rg for w in range(self.n_rg + 1)]

    def tile(self, x, n_kt):
        t = (max(0, x - ITEM) + self.gran // 2) // self.gran * self.gran
        return 0 if t < MIN else (n_kt if t > n_kt - MIN else t)

    def pieces(self, w):
        out = []
        if w >= self.n_rg:
            return out
        pos, end = self.bounds[w], self.bounds[w + 1]
        while pos < end:
            e = max(i for i in range(len(self.items)) if self.cum[i] <= pos)
            lo, hi = self.cum[e], self.cum[e + 1]
            assert lo <= pos < hi and self.items[e] is not None
            n_kt = self.items[e][3]
            x0, cut = pos - lo, hi > end
            t0 = self.tile(x0, n_kt) if x0 > 0 else 0
            t1 = self.tile(end - lo, n_kt) if cut else n_kt
            pos = end if cut else hi
            if n_kt == 0:
                if x0 == 0:
                    out.append((e, 0, 0, n_kt))
            elif t1 > t0:
                out.append((e, t0, t1, n_kt))
        return out


def check_queue(q):
    cover = {}
    part = {}    # (range, slot) -> (entry, t0, t1, n_kt)
    for w in range(q.n_wg):
        for e, t0, t1, n_kt in q.pieces(w):
            assert t0 % q.tpb == 0
            cover.setdefault(e, []).append((t0, t1))
            if (t0, t1) != (0, n_kt):
                slot = (w, 0 if t0 > 0 else 1)
                assert slot not in part
                part[slot] = (e, t0, t1, n_kt)
    assert sorted(cover) == [e for e, it in enumerate(q.items) if it is not None]
    for e, spans in cover.items():
        n_kt = q.items[e][3]
        assert spans[0][0] == 0 and spans[-1][1] == n_kt
        assert all(a[1] == b[0] for a, b in zip(spans, spans[1:]))
    for (w, slot), (e, t0, t1, n_kt) in part.items():    # the merge's walk
        if slot == 1:
            got, j = [(t0, t1)], w + 1
            while got[-1][1] < n_kt:
                p = part.get((j, 0))
                if p is not None:
                    assert p[0] == e
                    got.append(p[1:3])
                j += 1
                assert j <= q.n_wg
            assert got == cover[e]


SHAPES = [(8, 32, 64), (4, 32, 64), (2, 32, 64), (1, 32, 64), (16, 32, 64), (3, 32, 64), (8, 128, 64), (4, 32, 32)]


@pytest.mark.parametrize("n_y,rows,n_wg", SHAPES)
@pytest.mark.parametrize("tpb", [1, 2, 8, 32])
def test_ranges_cover_and_chain(n_y, rows, n_wg, tpb):
    rng = random.Random(n_y * 1000 + rows + tpb)
    for trial in range(6):
        n = rng.choice((1, 1, 2, 4, 7))
        lq = [rng.choice((0, 1, 5, rows, rows + 1, rng.randint(1, 1500))) for _ in range(n)]
        if not any(lq):
            lq[0] = 1
        lk = [x + rng.choice((0, 0, 37, 256, rng.randint(0, 9000))) for x in lq]
        if trial == 5:
            lk[0] = max(0, lq[0] - 50)    # rows without any visible key
        pin = n_y * n >= 8
        rep = 8 // n_y if n_y < 8 and 8 % n_y == 0 else 1
        if pin and cdiv(max(lq), rows) < 2 * rep:    # not enough query tiles to share
            rep = 1
        pin = pin or rep > 1
        for x in range(8) if pin else (0,):
            check_queue(Queue(x, lq, lk, n_y, rows, pin, rep, n_wg if pin else 8 * n_wg, tpb, trial != 4))


def would_cut(n, total_q, max_q, max_k, hq, hkv, d, kv):
    """Whether the library would cut such a launch: it asks for the partials' buffer, with nothing launched."""
    need = ctypes.c_int64()
    rc = lib().nq_varlen_prefill_split(None, 0, 0, None, None, 0, None, None, max_q, max_k, None, 0, 0, 0, None, 0, 0, n,
                                       hq, hkv, d, 256, 1.0, 1, dtype_code(torch.bfloat16), dtype_code(kv), None, None,
                                       None, 0, None, 0, 0, total_q, None, 0, need, None)
    assert rc == 1 and need.value > 0 or rc < 0 and need.value == 0
    return rc == 1


BF16, FP8 = torch.bfloat16, torch.float8_e4m3fn


@pytest.mark.parametrize("n,total_q,max_q,prefix,d,kv,cut", [
    (16, 3100, 300, 8192, 256, BF16, False),    # 1.7 items per workgroup of nearly one cost: they share K/V in L2
    (16, 3100, 300, 512, 256, BF16, False),
    (16, 3100, 300, 8192, 256, FP8, True),
    (16, 3100, 300, 8192, 128, BF16, True),
    (8, 3000, 600, 8192, 256, BF16, False),
    (4, 3300, 1111, 8192, 256, BF16, False),
    (4, 3300, 1111, 0, 256, BF16, True),        # causal from the first key: costs differ
    (12, 7668, 639, 0, 256, BF16, False),
    (4, 2400, 600, 8192, 256, BF16, True),      # 1.2 items
    (1, 3600, 3600, 8192, 256, BF16, True),     # one sequence
    (4, 800, 300, 6000, 256, BF16, True),
])
def test_which_launches_are_cut(n, total_q, max_q, prefix, d, kv, cut):
    hq, hkv = (16, 4) if d == 256 else (32, 8)
    hkv = 2 if n == 12 else hkv
    assert would_cut(n, total_q, max_q, max_q + prefix, 4 * hkv, hkv, d, kv) == cut
