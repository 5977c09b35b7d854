"""Work lists whose pairs or sizes take the plan's less common routes, through
the C-ABI, against numpy."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import block_amd
from capi import Device, check, lib, vp
from test_gpu_products import PAIR, VBLOCK, Chunk, reference, work_list

pytestmark = pytest.mark.gpu
lib.bsg_sigma_profile.restype = ctypes.c_int
lib.bsg_sigma_profile.argtypes = [vp, vp, vp, vp, vp, ctypes.c_int32, ctypes.c_int32, ctypes.c_int32] + [vp] * 3

BOTH = pytest.mark.parametrize("precision", [block_amd.FP64, block_amd.SPLIT_BF16], ids=["fp64", "split"])


class Plan:
    """A plan of one chunk and its operator arena on the device."""

    def __init__(self, d, vbs, prs, wave, arena, split=False):
        self.d, self.wave, self.h = d, wave, vp()
        chunk = Chunk(vbs.ctypes.data, len(vbs), prs.ctypes.data, len(prs))
        check(lib.bsg_plan_create(d.ctx, ctypes.byref(chunk), 1, wave, ctypes.byref(self.h)))
        self.arena, self.n = d.upload(arena), len(arena)
        if split:
            self.split()

    def split(self):
        check(lib.bsg_plan_split_arena(self.d.ctx, self.h, self.arena, self.n))

    def apply(self, c, precision, call=lib.bsg_sigma_apply):
        """H c for the rows of c in one call."""
        c = np.atleast_2d(c)
        dc, dv = self.d.upload(c), self.d.zeros(c.size)
        check(call(self.d.ctx, self.h, self.arena, dc, dv, len(c), precision))
        return self.d.download(dv, c.shape)

    def profile(self, c, precision, reps=2, nvec=1):
        """(wall ms, kernel ms, kernel launches of one application)"""
        dc, dv = self.d.upload(c), self.d.zeros(c.size)
        wall, ms, n = ctypes.c_double(), (ctypes.c_double * 3)(), (ctypes.c_long * 3)()
        check(lib.bsg_sigma_profile(self.d.ctx, self.h, self.arena, dc, dv, nvec, reps, precision, ctypes.byref(wall),
                                    ms, n))
        return wall.value, list(ms), n[0] // reps

    def __enter__(self):
        return self

    def __exit__(self, *a):
        lib.bsg_plan_destroy(self.h)


def tolerance(vbs, prs, precision):
    """Per sum of absolute products: each of a value's two nested sums of at
    most `deep` products rounds once per addition, on both sides of the
    comparison; split: operands rounded to 2^-24, the slice products left out
    about 3 x 2^-24, FP32 sums of 6 x 32 terms per K group (at most 6 + 32
    roundings), in each of the two products."""
    deep = 4 * max(int(prs["k1"].max() + prs["k2"].max()), int(vbs["count"].max()))
    tol = 2 * deep * np.finfo(float).eps
    return tol + 2 * (2 + 3 + 38) * 2.0 ** -24 if precision == block_amd.SPLIT_BF16 else tol


def agree(got, vbs, prs, c, arena, wave, precision):
    ref, bound = reference(vbs, prs, c, arena, wave)
    err = np.abs(got - ref)
    assert np.all(err <= tolerance(vbs, prs, precision) * bound), float((err / np.maximum(bound, 1e-300)).max())


@BOTH
@pytest.mark.parametrize("m,n", [(90, 100), (40, 50), (20, 24)])
def test_one_c_offset_as_different_shapes(m, n, precision):
    """Pairs that read the same C offset as blocks of different shapes (of the
    same and of different sizes)."""
    print(f"[gpu] one C offset, {m} x {n}, precision {precision}", flush=True)
    rng = np.random.default_rng(m)
    depths = [(66, 70), (70, 66), (3, 100), (100, 3), (17, 17), (m, 40), (40, n)]
    size = max(k1 * k2 for k1, k2 in depths)
    prs, arena = [], 0
    for k1, k2 in depths:
        a, b = (-1 if k1 == m else arena), (-1 if k2 == n else arena + m * k1)
        arena += m * k1 + k2 * n
        prs.append((a, 0, b, k1, k2, int(rng.integers(2)), int(rng.integers(2)), 1.0, rng.uniform(0.5, 1.5)))
    prs = np.array(prs, dtype=PAIR)
    vbs = np.array([(size, m, n, 0, len(prs))], dtype=VBLOCK)
    wave = size + m * n
    ops = rng.standard_normal(arena)
    c = np.zeros(wave)
    c[:size] = rng.standard_normal(size)
    with Device() as d, Plan(d, vbs, prs, wave, ops, precision == block_amd.SPLIT_BF16) as p:
        agree(p.apply(c, precision)[0], vbs, prs, c, ops, wave, precision)


@BOTH
@pytest.mark.parametrize("sides,depths,side", [
    ([(16, 9), (3, 16)], [(16, 5), (8, 16)], False),    # nothing beside the main stream
    ([(32, 25), (26, 32)], [(30, 5), (8, 27)], True),   # the widest small blocks alone
    ([(16, 9), (70, 66)], [(16, 5), (70, 66)], None),   # with blocks of another kernel
], ids=["to16", "to32", "mixed"])
def test_profile(sides, depths, side, precision):
    """The timing helper times every list; the side stream's time is there
    exactly if the list has kernels that run there (both identity partners are
    left out: split precision runs an identity A on another kernel)."""
    print(f"[gpu] profile {sides} precision {precision}", flush=True)
    rng = np.random.default_rng(3)
    vbs, prs, wave, _, arena = work_list(rng, sides, depths, 2)
    keep = (prs["a_off"] >= 0) & (prs["b_off"] >= 0)
    for vb in vbs:
        vb["count"] = keep[vb["first"]:vb["first"] + vb["count"]].sum()
    prs = prs[keep]
    vbs["first"] = np.concatenate([[0], np.cumsum(vbs["count"])[:-1]])
    with Device() as d, Plan(d, vbs, prs, wave, arena, precision == block_amd.SPLIT_BF16) as p:
        wall, ms, launches = p.profile(rng.standard_normal(wave), precision)
    assert wall > 0.0 and ms[0] > 0.0 and launches >= 1
    if side is not None:
        assert (ms[2] > 0.0) == side


@BOTH
def test_large_blocks_without_w(precision):
    """Large blocks whose pairs all have an identity partner and need no W:
    their product tiles are one launch, not one per block."""
    print(f"[gpu] large blocks without W, precision {precision}", flush=True)
    rng = np.random.default_rng(4)
    m, n, nb = 98, 103, 24
    prs, arena = [], 0
    for i in range(nb):
        c = i * m * n
        prs += [(arena, c, -1, m, n, i & 1, 0, -1.0, 0.75), (-1, c, -1, m, n, 0, 0, 1.0, 1.5)]
        arena += m * m
        if precision == block_amd.FP64:  # (split precision slices an identity A's W)
            prs.append((-1, c, arena, m, n, 0, i & 1, 1.0, -0.5))
            arena += n * n
    prs, per, size = np.array(prs, dtype=PAIR), len(prs) // nb, nb * m * n
    vbs = np.array([(size + i * m * n, m, n, per * i, per) for i in range(nb)], dtype=VBLOCK)
    ops, c = rng.standard_normal(arena), np.zeros(2 * size)
    c[:size] = rng.standard_normal(size)
    with Device() as d, Plan(d, vbs, prs, 2 * size, ops, precision == block_amd.SPLIT_BF16) as p:
        agree(p.apply(c, precision)[0], vbs, prs, c, ops, 2 * size, precision)
        launches = p.profile(c, precision)[2]
    # the products, split: the wavefunction's slices; units past one per block: their reduction
    assert launches <= 3


class Products:
    """V blocks of one shape with `count` pairs each, all pairs reading a few
    operators (in both storage orders) and C blocks, so that numpy sums long
    lists quickly."""

    def __init__(self, rng, m, n, depths, count, blocks=1, reuse=3):
        self.m, self.n = m, n
        self.blocks, self.wave, arena, self.ops = [], 0, [], 0

        def operator(rows, cols):
            x, off = rng.standard_normal((rows, cols)), self.ops
            arena.extend([x.ravel(), x.T.ravel()])
            self.ops += 2 * x.size
            return x, (off, off + x.size)

        sets = []
        for k1, k2 in depths:
            cs = []
            for _ in range(reuse):
                cs.append(self.wave)
                self.wave += k1 * k2
            sets.append((k1, k2, [operator(m, k1) for _ in range(reuse)], cs, [operator(k2, n) for _ in range(reuse)]))
        self.csize, self.terms, prs, vbs = self.wave, [], [], []
        for _ in range(blocks):
            first = len(prs)
            mine = {}
            for q in range(count):
                s = q % len(sets)
                k1, k2, a, c, b = sets[s]
                i, j, l = rng.integers(reuse, size=3)
                ta, tb = int(rng.integers(2)), int(rng.integers(2))
                al = float(rng.uniform(0.5, 1.5) * rng.choice([-1.0, 1.0]))
                prs.append((a[i][1][ta], c[j], b[l][1][tb], k1, k2, ta, tb, -1.0, al))
                x = mine.setdefault((s, i, j, l), [0.0, 0.0])
                x[0] -= al
                x[1] += abs(al)
            self.terms.append((self.wave, mine))
            vbs.append((self.wave, m, n, first, count))
            self.wave += m * n
        self.sets, self.arena = sets, np.concatenate(arena)
        self.vbs, self.prs = np.array(vbs, dtype=VBLOCK), np.array(prs, dtype=PAIR)

    def vectors(self, rng, nroot):
        c = np.zeros((nroot, self.wave))
        c[:, :self.csize] = rng.standard_normal((nroot, self.csize))
        return c

    def agree(self, got, c, precision):
        tol = tolerance(self.vbs, self.prs, precision)
        assert np.all(got[:self.csize] == 0.0)
        half = {}
        for s, (k1, k2, a, cs, _) in enumerate(self.sets):
            for j, o in enumerate(cs):
                x = c[o:o + k1 * k2].reshape(k1, k2)
                for i, (y, _) in enumerate(a):
                    half[s, i, j] = y @ x, np.abs(y) @ np.abs(x)
        for off, mine in self.terms:
            w = {}
            for (s, i, j, l), (f, g) in mine.items():
                x, y = half[s, i, j]
                z = w.setdefault((s, l), [np.zeros_like(x), np.zeros_like(x)])
                z[0] += f * x
                z[1] += g * y
            v = sum(z[0] @ self.sets[s][4][l][0] for (s, l), z in w.items())
            bound = sum(z[1] @ np.abs(self.sets[s][4][l][0]) for (s, l), z in w.items())
            err = np.abs(got[off:off + v.size].reshape(v.shape) - v)
            assert np.all(err <= tol * bound), float((err / bound).max())


def test_rounds_stay_within_the_scratch():
    """Product tiles in four rounds of almost half the W scratch each, whose
    last unit does not fit: the rounds stay within it, so that four roots
    still share each launch, and six roots take a second set of launches."""
    print("[gpu] rounds of product tiles within the W scratch", flush=True)
    rng = np.random.default_rng(5)
    # 16 pairs of 128,000 doubles of W are a unit; four rounds of 2^26 doubles hold 2097 pairs
    x = Products(rng, 1000, 101, [(99, 128)], 2096)
    c = x.vectors(rng, 6)
    with Device() as d, Plan(d, x.vbs, x.prs, x.wave, x.arena) as p:
        one = np.concatenate([p.apply(v, block_amd.FP64) for v in c])
        single = p.profile(c[0], block_amd.FP64)[2]
        check(lib.bsg_plan_set_batch(d.ctx, p.h, 4))
        four = p.profile(c[:4], block_amd.FP64, nvec=4)[2]
        assert np.array_equal(p.apply(c[:4], block_amd.FP64), one[:4])
        check(lib.bsg_plan_set_batch(d.ctx, p.h, 6))
        six = p.profile(c, block_amd.FP64, nvec=6)[2]
        assert np.array_equal(p.apply(c, block_amd.FP64), one)
    for v, w in zip(one, c):
        x.agree(v, w, block_amd.FP64)
    print(f"[gpu] launches: one root {single}, four {four}, six {six}", flush=True)
    assert four == single
    assert single < six <= 2 * single


def test_w_scratch_is_kept_for_the_next_plan():
    """Four roots' W scratch (1 to 4 GB) stays with the context when its plan
    goes, serves the next plan, smaller or as large, and is given back with the
    context."""
    print("[gpu] W scratch kept", flush=True)
    rng = np.random.default_rng(6)
    x = Products(rng, 1000, 101, [(99, 128)], 600)
    c = x.vectors(rng, 4)
    gb = 1 << 30

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info(0)[0]

    with Device() as d, Plan(d, x.vbs, x.prs, x.wave, x.arena) as p:  # what the library holds until the process ends
        p.apply(c[0], block_amd.FP64)
    start = free()
    with Device() as d:
        got = []
        for i in range(3):
            with Plan(d, x.vbs, x.prs, x.wave, x.arena) as p:
                before = free()
                check(lib.bsg_plan_set_batch(d.ctx, p.h, 4))
                assert i == 0 or before - free() < gb // 4
                got.append(p.apply(c, block_amd.FP64))
            assert gb < start - free() < 5 * gb
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    assert start - free() < gb // 4
    for v, w in zip(got[0], c):
        x.agree(v, w, block_amd.FP64)


@BOTH
def test_two_threads_apply_two_plans_of_one_context(precision):
    """Applications of two plans from two threads, whose large blocks share
    the context's W scratch, each in order and as alone."""
    print(f"[gpu] two threads, one context, precision {precision}", flush=True)
    rng = np.random.default_rng(8)
    xs = [Products(rng, 130, 101, [(99, 128)], 40, blocks=6), Products(rng, 97, 140, [(120, 103)], 40, blocks=6)]
    cs = [x.vectors(rng, 1) for x in xs]
    reps = 40
    with Device() as d:
        plans = [Plan(d, x.vbs, x.prs, x.wave, x.arena, precision == block_amd.SPLIT_BF16) for x in xs]
        one = [p.apply(c, precision)[0] for p, c in zip(plans, cs)]
        dc = [d.upload(c) for c in cs]
        dv = [[d.zeros(x.wave) for _ in range(reps)] for x in xs]
        rcs = [[], []]

        def work(i):
            for v in dv[i]:
                rcs[i].append(lib.bsg_sigma_apply(d.ctx, plans[i].h, plans[i].arena, dc[i], v, 1, precision))

        threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert rcs == [[0] * reps] * 2
        for i, x in enumerate(xs):
            for v in dv[i]:
                assert np.array_equal(d.download(v, x.wave), one[i])
            plans[i].__exit__()
    for x, v, c in zip(xs, one, cs):
        x.agree(v, c[0], precision)


@pytest.mark.parametrize("m,n,depths,count,blocks", [
    (32, 32, [(1, 1)], 1000, 30),                    # cut finely, as a superblock of little work
    (40, 45, [(1, 1), (60, 3), (90, 1)], 1000, 30),  # in three panel classes as well
    (60, 64, [(8, 8), (50, 5), (90, 3)], 3, 4000),   # one pair in each class of every block
    (16, 16, [(8, 8), (20, 5), (30, 3), (40, 3)], 4, 12000),
], ids=["fine", "fine_classes", "classes", "small_classes"])
def test_allocation_free_call_takes_lists_of_many_small_units(m, n, depths, count, blocks):
    """Lists whose partial tiles fit the static scratch when cut at fixed costs
    fit it as they are cut, in both precisions."""
    print(f"[gpu] allocation-free, {blocks} blocks of {m} x {n}", flush=True)
    rng = np.random.default_rng(m)
    x = Products(rng, m, n, depths, count, blocks)
    c = x.vectors(rng, 1)
    with Device() as d, Plan(d, x.vbs, x.prs, x.wave, x.arena, True) as p:
        for precision in (block_amd.FP64, block_amd.SPLIT_BF16):
            got = p.apply(c, precision, lib.bsg_sigma_apply_noalloc)
            assert np.array_equal(got, p.apply(c, precision))
            x.agree(got[0], c[0], precision)


def test_partial_doubles_cover_split_precision_from_the_start():
    """The partial tiles a plan reports are those of both precisions, before
    the split set-up as after it."""
    print("[gpu] partial tiles before the split set-up", flush=True)
    rng = np.random.default_rng(10)
    for m, n, depths in ((40, 50, [(45, 47)]), (20, 24, [(9, 24), (33, 40)]), (90, 70, [(80, 85), (3, 100)])):
        x = Products(rng, m, n, depths, 300, blocks=4)
        with Device() as d, Plan(d, x.vbs, x.prs, x.wave, x.arena) as p, Plan(d, x.vbs, x.prs, x.wave, x.arena) as q:
            before = lib.bsg_plan_partial_doubles(p.h)
            p.split()
            q.split()
            assert before == lib.bsg_plan_partial_doubles(p.h) == lib.bsg_plan_partial_doubles(q.h) > 0


@BOTH
def test_two_rounds_of_odd_sizes(precision):
    """More W than one round holds: two rounds, each in its half of the
    scratch on its own stream, with odd sizes, several units per block and a
    block of identity partners among them."""
    print(f"[gpu] two rounds, precision {precision}", flush=True)
    rng = np.random.default_rng(11)
    x = Products(rng, 99, 131, [(97, 103), (101, 129), (3, 111), (120, 1)], 700, blocks=2)
    # past 2^23 doubles of W; the split ones are three quarters of that and padded
    w = sum(99 * int(k2) for k2 in x.prs["k2"])
    assert w * 3 / 4 > 1 << 23
    c = x.vectors(rng, 3)
    with Device() as d, Plan(d, x.vbs, x.prs, x.wave, x.arena, precision == block_amd.SPLIT_BF16) as p:
        one = np.concatenate([p.apply(v, precision) for v in c])
        check(lib.bsg_plan_set_batch(d.ctx, p.h, 2))
        assert np.array_equal(p.apply(c, precision), one)
    for v, u in zip(one, c):
        x.agree(v, u, precision)


def test_wide_split_tiles_at_odd_sizes():
    """Enough W tiles for the 128 x 128 split tiles, next to 64 x 64 ones where
    those would pad too much, at odd sizes around both."""
    print("[gpu] wide split tiles", flush=True)
    rng = np.random.default_rng(12)
    lists = [Products(rng, m, n, [(k, 121), (k, 127), (7, 129), (129, 70)], 2600, blocks=1)
             for m, n, k in ((125, 127, 113), (129, 97, 31), (257, 115, 66), (65, 250, 125))]
    # one list of all: C blocks, operators and V blocks of the parts one after the other
    vbs, prs, arena, first, woff, aoff = [], [], [], 0, 0, 0
    for x in lists:
        v, p = x.vbs.copy(), x.prs.copy()
        v["v_off"] += woff
        v["first"] += first
        for f in ("a_off", "b_off"):
            p[f] += aoff
        p["c_off"] += woff
        vbs.append(v)
        prs.append(p)
        arena.append(x.arena)
        first, woff, aoff = first + len(p), woff + x.wave, aoff + len(x.arena)
    vbs, prs, arena = np.concatenate(vbs), np.concatenate(prs), np.concatenate(arena)
    tiles = sum(-(-int(v["m"]) // 128) * sum(-(-prs["k2"][v["first"]:v["first"] + v["count"]] // 128)) for v in vbs)
    assert tiles >= 1 << 14
    c = np.concatenate([x.vectors(rng, 1)[0] for x in lists])
    with Device() as d, Plan(d, vbs, prs, woff, arena, True) as p:
        got = p.apply(c, block_amd.SPLIT_BF16)[0]
    o = 0
    for x in lists:
        x.agree(got[o:o + x.wave], c[o:o + x.wave], block_amd.SPLIT_BF16)
        o += x.wave


CANDIDATES = [(p, i) for p in (block_amd.FP64, block_amd.SPLIT_BF16) for i in range(block_amd.tile_candidates(p))]


@pytest.mark.parametrize("precision,cand", CANDIDATES, ids=[f"{'split' if p else 'fp64'}{i}" for p, i in CANDIDATES])
def test_every_tile_candidate(precision, cand):
    """Every candidate a tile table may name (grouped tiles, wide ones of four
    and eight wavefronts, per-wave tiles), for all V blocks, with blocks wider
    than each of their tiles."""
    print(f"[gpu] tile candidate {cand} of precision {precision}", flush=True)
    rng = np.random.default_rng(13)
    shapes, depths = [(33, 35), (64, 48), (70, 129), (17, 257), (35, 390), (20, 775)], [(1, 2), (37, 45), (66, 70), (90, 33)]
    vbs, prs, wave, wave_c, arena = work_list(rng, shapes, depths, 2)
    c = np.zeros(wave)
    c[:wave_c] = rng.standard_normal(wave_c)
    split = precision == block_amd.SPLIT_BF16
    try:
        block_amd.set_tile_table([(1, 1 << 20, 1, 1 << 20, -1 if split else cand, cand if split else -1)])
        with Device() as d, Plan(d, vbs, prs, wave, arena, split) as p:
            got = p.apply(c, precision)[0]
    finally:
        block_amd.set_tile_table(block_amd.read_tile_table())
    agree(got, vbs, prs, c, arena, wave, precision)


def test_a_refused_allocation_leaves_the_plan_usable():
    """More roots than memory holds: refused, the plan is as it was and its next
    applications succeed."""
    print("[gpu] refused batch", flush=True)
    rng = np.random.default_rng(14)
    x = Products(rng, 100, 60, [(40, 50)], 400, blocks=3)
    c = x.vectors(rng, 2)
    with Device() as d, Plan(d, x.vbs, x.prs, x.wave, x.arena) as p:
        one = p.apply(c, block_amd.FP64)
        assert 8 * lib.bsg_plan_partial_doubles(p.h) << 26 > 1 << 42  # 4 TB
        assert lib.bsg_plan_set_batch(d.ctx, p.h, 1 << 26) == -3  # BSG_ERR_NOMEM
        assert np.array_equal(p.apply(c, block_amd.FP64), one)
        check(lib.bsg_plan_set_batch(d.ctx, p.h, 2))
        assert np.array_equal(p.apply(c, block_amd.FP64), one)
