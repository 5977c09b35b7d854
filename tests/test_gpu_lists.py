"""Work lists whose pairs or sizes take the plan's less common routes, through
the C-ABI, against numpy."""
import ctypes

import numpy as np
import pytest

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

    def profile(self, c, precision, reps=2):
        """(wall ms, kernel ms, kernel launches of one application)"""
        dc, dv = self.d.upload(c), self.d.zeros(c.size)
        wall, ms, n = ctypes.c_double(), (ctypes.c_double * 3)(), (ctypes.c_long * 3)()
        check(lib.bsg_sigma_profile(self.d.ctx, self.h, self.arena, dc, dv, 1, reps, precision, ctypes.byref(wall),
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
