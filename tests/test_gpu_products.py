"""Sigma of hand-made work lists, FP64 and split precision, against numpy: V blocks and contraction
depths at the edges of the kernels' tiles (one row or column more or less than
a tile, odd depths, depths of one), every storage order of the operator
blocks, identity partners on either side, several units per V block, several
roots; through the C-ABI."""
import ctypes

import numpy as np
import pytest

import block_amd
from capi import Device, check, lib, vp

pytestmark = pytest.mark.gpu

PAIR = np.dtype([("a_off", "i8"), ("c_off", "i8"), ("b_off", "i8"), ("k1", "i4"), ("k2", "i4"), ("a_trans", "i4"),
                 ("b_trans", "i4"), ("alpha_a", "f8"), ("alpha", "f8")])
VBLOCK = np.dtype([("v_off", "i8"), ("m", "i4"), ("n", "i4"), ("first", "i4"), ("count", "i4")])


class Chunk(ctypes.Structure):
    _fields_ = [("vblocks", vp), ("n_vblocks", ctypes.c_int32), ("pairs", vp), ("n_pairs", ctypes.c_int32)]


for _name, _args in (("bsg_plan_create", [vp, vp, ctypes.c_int32, ctypes.c_int64, ctypes.POINTER(vp)]),
                     ("bsg_plan_destroy", [vp]), ("bsg_plan_set_batch", [vp, vp, ctypes.c_int32]),
                     ("bsg_plan_split_arena", [vp, vp, vp, ctypes.c_int64])):
    getattr(lib, _name).argtypes = _args
    getattr(lib, _name).restype = ctypes.c_int


def work_list(rng, shapes, depths, repeats):
    """V blocks of the given shapes; each has, per (k1, k2), the pairs of all
    storage orders of two operators, `repeats` times, and the pairs with an
    identity on the left, on the right and on both sides.  Returns (V blocks,
    pairs, wavefunction size, arena)."""
    coffs, off = {}, 0
    for m, n in shapes:
        for k in [(m, n)] + [(k1, n) for k1, _ in depths] + [(m, k2) for _, k2 in depths] + list(depths):
            if k not in coffs:
                coffs[k] = off
                off += k[0] * k[1]
    wave_c = off
    vbs, prs, arena = [], [], 0

    def pair(m, n, k1, k2, a, b):
        nonlocal arena
        ao, bo = -1, -1
        if a >= 0:
            ao, arena = arena, arena + m * k1
        if b >= 0:
            bo, arena = arena, arena + k2 * n
        prs.append((ao, coffs[(k1, k2)], bo, k1, k2, max(a, 0), max(b, 0), rng.choice([-1.0, 1.0]) if a >= 0 else 1.0,
                    rng.uniform(0.5, 1.5)))

    for m, n in shapes:
        first = len(prs)
        for _ in range(repeats):
            for k1, k2 in depths:
                for a in (0, 1):
                    for b in (0, 1):
                        pair(m, n, k1, k2, a, b)
        for k1, k2 in depths:
            pair(m, n, m, k2, -1, 0)
            pair(m, n, m, k2, -1, 1)
            pair(m, n, k1, n, 0, -1)
            pair(m, n, k1, n, 1, -1)
        pair(m, n, m, n, -1, -1)
        vbs.append((off, m, n, first, len(prs) - first))
        off += m * n
    return (np.array(vbs, dtype=VBLOCK), np.array(prs, dtype=PAIR), off, wave_c,
            rng.standard_normal(max(1, arena)))


def reference(vbs, prs, c, arena, wave):
    """H c and, elementwise, the sum of the absolute products (for the error
    bound)."""
    out, bound = np.zeros(wave), np.zeros(wave)
    for vb in vbs:
        m, n = int(vb["m"]), int(vb["n"])
        v, w = np.zeros((m, n)), np.zeros((m, n))
        for p in prs[vb["first"]:vb["first"] + vb["count"]]:
            k1, k2 = int(p["k1"]), int(p["k2"])
            x = c[p["c_off"]:p["c_off"] + k1 * k2].reshape(k1, k2)
            f, ax = p["alpha"], np.abs(x)
            if p["a_off"] >= 0:
                a = arena[p["a_off"]:p["a_off"] + m * k1]
                a = a.reshape(k1, m).T if p["a_trans"] else a.reshape(m, k1)
                x, ax, f = a @ x, np.abs(a) @ ax, f * p["alpha_a"]
            if p["b_off"] >= 0:
                b = arena[p["b_off"]:p["b_off"] + k2 * n]
                b = b.reshape(n, k2).T if p["b_trans"] else b.reshape(k2, n)
                x, ax = x @ b, ax @ np.abs(b)
            v += f * x
            w += abs(f) * ax
        o = int(vb["v_off"])
        out[o:o + m * n], bound[o:o + m * n] = v.ravel(), w.ravel()
    return out, bound


CASES = {
    # small-block kernel's V blocks with pairs it does not take, and the first
    # sizes above it
    "small": ([(1, 1), (16, 33), (33, 7), (32, 32), (17, 1)], [(1, 1), (40, 3), (5, 47), (33, 33)], 2),
    # up to 80 on a side
    "medium": ([(33, 34), (48, 49), (64, 17), (65, 64), (79, 80), (80, 33)], [(1, 2), (15, 17), (48, 33), (80, 79)], 2),
    # one side or one depth past 80
    "mixed": ([(81, 16), (40, 81), (33, 95), (64, 40)], [(81, 3), (7, 82), (96, 81), (30, 40)], 2),
    # 64-wide tiles: exact, one less, one more, depths of odd and even length
    "large": ([(127, 129), (128, 64), (97, 193), (191, 82)], [(1, 1), (2, 15), (16, 17), (129, 31), (100, 130)], 2),
    # small-block kernel: each of its width and depth classes (8s and 16s, one
    # less, one more), runs on one C block longer than its operand sets
    "width32": ([(1, 1), (8, 7), (16, 16), (17, 3), (9, 24), (24, 24), (25, 8), (32, 31)],
                [(1, 1), (8, 8), (9, 2), (3, 16), (17, 24), (24, 23), (25, 8), (31, 32)], 3),
    # many pairs per V block: several units, reduced in order
    "units": ([(90, 100), (50, 60), (20, 24)], [(61, 67), (24, 24)], 60),
}


@pytest.mark.parametrize("precision", [block_amd.FP64, block_amd.SPLIT_BF16], ids=["fp64", "split"])
@pytest.mark.parametrize("name", list(CASES))
def test_products(name, precision):
    print(f"[gpu] products {name} precision {precision}", flush=True)
    shapes, depths, repeats = CASES[name]
    rng = np.random.default_rng(sorted(CASES).index(name) + 5)
    vbs, prs, wave, wave_c, arena = work_list(rng, shapes, depths, repeats)
    nroot = 3
    c = np.zeros((nroot, wave))
    c[:, :wave_c] = rng.standard_normal((nroot, wave_c))
    with Device() as d:
        chunk = Chunk(vbs.ctypes.data, len(vbs), prs.ctypes.data, len(prs))
        plan = vp()
        check(lib.bsg_plan_create(d.ctx, ctypes.byref(chunk), 1, wave, ctypes.byref(plan)))
        try:
            da, dc = d.upload(arena), d.upload(c)
            dv = d.zeros(nroot * wave)
            if precision == block_amd.SPLIT_BF16:
                check(lib.bsg_plan_split_arena(d.ctx, plan, da, len(arena)))
            for r in range(nroot):  # one root at a time
                check(lib.bsg_sigma_apply(d.ctx, plan, da, dc.value + 8 * r * wave, dv.value + 8 * r * wave, 1,
                                          precision))
            one = d.download(dv, (nroot, wave))
            check(lib.bsg_plan_set_batch(d.ctx, plan, 2))
            check(lib.bsg_memset_zero(d.ctx, dv, 8 * nroot * wave))
            check(lib.bsg_sigma_apply(d.ctx, plan, da, dc, dv, nroot, precision))  # 2 + 1
            assert np.array_equal(d.download(dv, (nroot, wave)), one)
            check(lib.bsg_sigma_apply(d.ctx, plan, da, dc, dv, nroot, precision))  # accumulates
            twice = d.download(dv, (nroot, wave))
        finally:
            lib.bsg_plan_destroy(plan)
    eps = np.finfo(float).eps
    for r in range(nroot):
        ref, bound = reference(vbs, prs, c[r], arena, wave)
        # each of a value's two nested sums of at most `deep` products rounds
        # once per addition, on both sides of the comparison
        deep = 4 * max(int(prs["k1"].max() + prs["k2"].max()), int(vbs["count"].max()))
        tol = 2 * deep * eps
        if precision == block_amd.SPLIT_BF16:
            # per product of the two: operands rounded to 2^-24, the slice
            # products left out about 3 x 2^-24, FP32 sums of 6 x 32 terms in a
            # tree or chain per K group (at most 6 + 32 roundings on its result)
            tol += 2 * (2 + 3 + 38) * 2.0 ** -24
        err = np.abs(one[r] - ref)
        assert np.all(err <= tol * bound), (r, float((err / np.maximum(bound, 1e-300)).max()))
        assert np.all(np.abs(twice[r] - 2 * ref) <= 2 * tol * bound)
        assert np.all(one[r][:wave_c] == 0.0)  # nothing written outside the V blocks
