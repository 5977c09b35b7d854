"""Composite operators built in HBM (the block (x) dot recursions of
Operators.C:624-691,1059-1196,1472-1616,1905-1966,2322-2395 through
TensorProduct, operatorfunctions.C:146-254, as recorded scaled block copies
executed by bsg_build_apply) against the host build of the same operators,
and sweeps whose blocks never leave HBM against host-built sweeps."""
import ctypes

import numpy as np
import pytest

import block_amd
from capi import Device, check, lib, vp
from helpers import config_fcidump, random_fcidump

pytestmark = pytest.mark.gpu
lib.bsg_build_apply.argtypes = [vp, vp, ctypes.c_int32, vp, ctypes.c_int32]
lib.bsg_build_apply.restype = ctypes.c_int
COLS = block_amd.SWEEP_COLS


@pytest.mark.parametrize("name,nsys,M", [("hubbard12", 4, 40), ("syn16", 6, 60), ("syn16d2h", 6, 60)])
def test_device_build_matches_host_build(name, nsys, M):
    """Normal and complementary operator sets of sys (x) dot and sys (x)
    dot's complementary operators in its own basis, from a host block and
    from a device-only one: the same elements as the host build (the device
    sums every element's terms in the host's order, so they agree bitwise)."""
    print(f"[gpu] device build {name}", flush=True)
    ints = {"hubbard12": lambda: config_fcidump("hubbard12"),
            "syn16": lambda: random_fcidump(16, 21),
            "syn16d2h": lambda: random_fcidump(16, 22, d2h=True)}[name]()
    worst, n = block_amd.build_check(ints, nsys, M)
    print(f"[gpu] {name}: {n} operators, max |host - device| = {worst:.3e}", flush=True)
    assert n > 20
    assert worst <= 1e-14


def test_device_blocks_sweep_matches_host_blocks():
    """The same sweeps with blocks kept in HBM and with host-built blocks:
    the same energies (to 1e-12) and sigma counts per sweep."""
    print("[gpu] device-block sweep", flush=True)
    ints = random_fcidump(12, 31)
    sched = [(0, 40, 1e-8, 1e-5), (2, 80, 1e-11, 0.0)]
    e_d, sw_d = block_amd.dmrg(ints, schedule=sched, max_sweeps=4, sweep_tol=0.0, device_blocks=True)
    e_h, sw_h = block_amd.dmrg(ints, schedule=sched, max_sweeps=4, sweep_tol=0.0, device_blocks=False)
    np.testing.assert_allclose(sw_d[:, COLS.index("E0")], sw_h[:, COLS.index("E0")], rtol=0, atol=1e-12)
    assert np.array_equal(sw_d[:, COLS.index("sigma_calls")], sw_h[:, COLS.index("sigma_calls")])
    assert abs(e_d[0] - e_h[0]) <= 1e-12


@pytest.mark.parametrize("rows,cols,groups,deep", [(1, 1, 700, 1), (1, 3, 90, 2), (9, 8, 3000, 24), (300, 70, 3, 3)])
def test_rectangle_sizes(rows, cols, groups, deep):
    """Groups of every size up to rows x cols (a wavefront's elements may span
    64 groups or a part of one), up to `deep` sources each; against the sum
    in list order.  One rounding per product and sum on both sides, so the same
    bits."""
    print(f"[gpu] build of {groups} groups up to {rows} x {cols}", flush=True)
    rng = np.random.default_rng(rows * 1000 + cols)
    group = np.zeros(groups, dtype=[("dst", "i8"), ("ld", "i4"), ("rows", "i4"), ("cols", "i4"), ("first", "i4"),
                                    ("count", "i4"), ("pad", "i4")])
    group["rows"], group["cols"] = rng.integers(1, rows + 1, groups), rng.integers(1, cols + 1, groups)
    group["ld"] = group["cols"] + rng.integers(0, 3, groups)
    group["count"] = rng.integers(0, deep + 1, groups)
    if deep == 24:
        group["count"] = 24
        group["first"] = 24 * rng.permutation(groups)
    else:
        group["first"] = np.concatenate([[0], np.cumsum(group["count"])[:-1]])
    start = np.concatenate([[0], np.cumsum(group["rows"] * group["ld"])])
    nsrc = max(1, int(group["count"].sum()))
    source = np.zeros(nsrc, dtype=[("src", "i8"), ("ld", "i4"), ("trans", "i4"), ("alpha", "f8"), ("beta", "f8")])
    old = rng.standard_normal(rows * cols * 4 + 64)
    source["trans"], source["alpha"], source["beta"] = rng.integers(0, 2, nsrc), rng.standard_normal(nsrc), rng.standard_normal(nsrc)
    off = rng.integers(0, len(old) - rows * cols, nsrc)
    before = rng.standard_normal(int(start[-1]))
    sums = np.zeros(len(before))
    for i, g in enumerate(group):
        m, n = int(g["rows"]), int(g["cols"])
        total = np.zeros((m, n))
        for j in range(int(g["first"]), int(g["first"] + g["count"])):
            s = source[j]
            s["ld"] = m if s["trans"] else n
            a = old[off[j]:off[j] + m * n]
            total += (s["alpha"] * (a.reshape(n, m).T if s["trans"] else a.reshape(m, n))) * s["beta"]
        np.lib.stride_tricks.as_strided(sums[start[i]:], (m, n), (8 * int(g["ld"]), 8))[:] = total
    source["ld"][source["ld"] == 0] = 1
    with Device() as d:
        dold, ddst = d.upload(old), d.upload(before)
        group["dst"], source["src"] = ddst.value + 8 * start[:-1], dold.value + 8 * off
        for _ in range(2):
            check(lib.bsg_build_apply(d.ctx, group.ctypes.data, groups, source.ctypes.data, nsrc))
        got = d.download(ddst, before.shape)
    assert np.array_equal(got, (before + sums) + sums)
