"""Which superblocks the precision ladder's split phase runs on."""
import pytest

import block_amd
from helpers import config_fcidump, random_fcidump

pytestmark = pytest.mark.gpu


def test_ladder_skips_superblocks_that_split_precision_slows_down():
    """Blocks up to 96 run faster in FP64, though split precision would put
    most of their flops on BF16 slices: a sweep over such superblocks makes no
    split application unless it is told to."""
    print("[gpu] ladder on blocks up to 96", flush=True)
    ints = random_fcidump(12, 31)
    sched = [(0, 60, 1e-6, 1e-5), (1, 100, 1e-9, 0.0)]
    runs = {}
    for name, kw in {"fp64": {}, "ladder": dict(ladder=1e-5), "told": dict(ladder=1e-5, ladder_min_share=0.0)}.items():
        e, sw = block_amd.dmrg(ints, schedule=sched, max_sweeps=3, sweep_tol=0.0, **kw)
        runs[name] = e[0], sw[:, block_amd.SWEEP_COLS.index("split_calls")].sum()
    print(f"[gpu] split calls {runs['ladder'][1]:.0f}, told to {runs['told'][1]:.0f}", flush=True)
    assert runs["ladder"][1] == runs["fp64"][1] == 0 < runs["told"][1]
    assert runs["ladder"][0] == runs["fp64"][0]
    assert abs(runs["told"][0] - runs["fp64"][0]) <= 1e-8


def test_gain_share():
    """Share of the flops in pairs with a side or depth past 96: none where no
    V block passes 96 (nor a depth, which is another block's side), most of them
    where the blocks are hundreds wide."""
    print("[gpu] split gain share", flush=True)
    small = block_amd.SuperBlock(random_fcidump(16, 21), 16, 0, 0, 7, 200)
    assert 32 < max(max(s) for s in small.block_shapes()) <= 96
    h = block_amd.multiply_h(small)
    assert h.split_gain_share == 0.0 and h.split_share > 0.5
    wide = block_amd.SuperBlock.from_dmrg_warmup(config_fcidump("syn24"), 24, 0, 0, 500)
    h = block_amd.multiply_h(wide)
    assert 0.5 < h.split_gain_share <= 1.0
