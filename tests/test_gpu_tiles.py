"""PPM sweep tiles: the fused sweep (face values through LDS; along j and k
a wave holds `seg` cells along the axis by 64 / seg consecutive i) against
the split form (face values through
HBM from their own kernel), bit for bit: state, time, counters and the
stored fluxes, for 2D and 3D tori, one stored phi row, FP64 and mixed,
segment lengths that do and do not divide the extents, alone and in a
batch."""
from dataclasses import replace

import numpy as np
import pytest

from raishinsource_amd import configs, native

pytestmark = pytest.mark.gpu


def bitdiff(a, b):
    a = np.ascontiguousarray(a)
    b = np.ascontiguousarray(b)
    both_nan = np.isnan(a) & np.isnan(b)
    return int(np.count_nonzero((a.view(np.uint64) != b.view(np.uint64)) & ~both_nan))


def make(p, mixed=False, seed=0):
    p = p.resolved()
    g = native.setup_grid(p)
    m = native.setup_metric(p, g)
    uri = native.setup_torus(p, g, m, seed=seed, noise=0.02)
    mod = native.Model(p, g, m)
    mod.set_state(uri)
    mod.set_precision(mixed)
    return mod


def same(a, b, tag):
    wa, ua, ta = a.get_state()
    wb, ub, tb = b.get_state()
    assert ta == tb, tag
    assert bitdiff(wa, wb) == 0 and bitdiff(ua, ub) == 0, tag
    assert a.counters() == b.counters(), tag
    fa, ca = a.fluxes()
    fb, cb = b.fluxes()
    assert bitdiff(fa, fb) == 0 and bitdiff(ca, cb) == 0, tag


CASES = [
    ("t3dppm", False, (1, 0, 0), (0, 8, 16)),
    ("t3dppm", True, (1, 0, 0), (0, 64, 4)),
    ("uppm", False, (1, 0, 0), (0, 2, 32)),
    ("uppm", True, (1, 0, 0), (0, 0, 0)),
    ("c1", False, (1, 0, 0), (0, 16, 8)),      # one stored phi row
    ("t2d", True, (1, 0, 0), (0, 4, 64)),      # one stored phi row, mixed
]


@pytest.mark.parametrize("name,mixed,ta,tb", CASES)
def test_fused_sweep_equals_split(name, mixed, ta, tb):
    a, b = make(configs.ALL[name], mixed), make(configs.ALL[name], mixed)
    a.set_sweep_tiles(*ta)
    b.set_sweep_tiles(*tb)
    assert a.sweep_tiles()["ppm_split"] == ta[0] and b.sweep_tiles()["ppm_split"] == tb[0]
    for s in range(3):
        assert a.step(1) == b.step(1), s
    same(a, b, "eager")
    a.step_graph(1)
    b.step_graph(1)
    same(a, b, "graph")
    a.close()
    b.close()


def test_fused_sweep_in_a_batch():
    # RK2 members (a batch's members make the same launch sequence)
    ps = [configs.T2D, configs.U_PPM, replace(configs.T3D_PPM, name="t3dppm_b", jmax=20, irkt=2)]
    alone = [make(p, q == 1, seed=q) for q, p in enumerate(ps)]
    batched = [make(p, q == 1, seed=q) for q, p in enumerate(ps)]
    for q, mm in enumerate(alone):
        mm.set_sweep_tiles(1, 0, 0)
    for q, mm in enumerate(batched):
        mm.set_sweep_tiles(0, 4 << q, 32 >> q)
    for mm in alone:
        mm.step(4)
    b = native.Batch(batched)
    b.step(1)
    b.step_graph(1)
    b.step(1)
    for x, y in zip(alone, batched):
        same(x, y, "batch")
    b.set([])
    b.close()
    for mm in alone + batched:
        mm.close()


def test_autotuner_picks_tiles():
    p = configs.T3D_PPM.resolved()
    g = native.setup_grid(p)
    m = native.setup_metric(p, g)
    uri = native.setup_torus(p, g, m, seed=0, noise=0.02)
    ref = native.Model(p, g, m)
    ref.set_state(uri)
    mod = native.Model(p, g, m)
    tuned = mod.autotune(uri, steps=1)
    print("tuned", tuned)
    assert tuned["ppm_split"] == 0 and tuned["seg_j"] in (8, 16, 32) and tuned["seg_k"] in (8, 16, 32)
    with pytest.raises(native.RaishinError, match="power of two"):
        mod.set_sweep_tiles(0, 6, 8)
    ref.step(3)
    mod.step(3)
    same(ref, mod, "tuned")
    ref.close()
    mod.close()


@pytest.mark.parametrize("threads", [64, 128, 192, 256])
@pytest.mark.parametrize("ni,nj,nk,seg,mixed", [(17, 11, 15, 0, False), (72, 13, 30, 0, True), (75, 16, 71, 8, False)])
def test_workgroup_tiles_equal_split(threads, ni, nj, nk, seg, mixed):
    """The sweeps' workgroup tiles (rows of a workgroup or of 16, 32, 64
    lanes along i; stacked waves along j and k) at extents one below, at and
    above what a tile covers, against the split form."""
    p = configs.Pram("tile", ni, nj, nk, irec=5, irkt=3, cfl=0.4)
    a, b = make(p, mixed), make(p, mixed)
    a.set_sweep_tiles(1, 0, 0)
    b.set_block_sizes([threads] * 8)
    b.set_sweep_tiles(0, seg, seg)
    for s in range(2):
        assert a.step(1) == b.step(1), s
    same(a, b, threads)
    a.close()
    b.close()


@pytest.mark.parametrize("name,mixed,threads", [("t2d", False, 256), ("t2d", True, 64), ("t3dppm", False, 128)])
def test_one_launch_equals_separate(name, mixed, threads):
    """The three sweeps, the CFL reduction and its combination in the
    launches of a stage against a launch each (a model whose kernels are
    timed), with the same time and step."""
    a, b = make(configs.ALL[name], mixed), make(configs.ALL[name], mixed)
    for mm in (a, b):
        mm.set_block_sizes([threads] * 8)
    b.set_timing(True)
    for s in range(3):
        assert a.step(1) == b.step(1), s
    assert b.get_timing()["sweep_k"][1] > 0 and b.get_timing()["cfl"][1] == 3
    same(a, b, name)
    a.close()
    b.close()


@pytest.mark.parametrize("name,mixed,threads", [("umc", False, 64), ("uleis", True, 256), ("ump5", False, 128),
                                                ("uweno", False, 256), ("t2dmc", False, 192)])
def test_one_launch_of_other_sweeps(name, mixed, threads):
    """As test_one_launch_equals_separate for MC, MP5 and WENO5, against the
    same model in a batch too (a launch per sweep there)."""
    a, b, c = (make(configs.ALL[name], mixed) for _ in range(3))
    for mm in (a, b, c):
        mm.set_block_sizes([threads] * 8)
    b.set_timing(True)
    batch = native.Batch([c])
    for s in range(2):
        assert np.array_equal(a.step(1), b.step(1), equal_nan=True), s
    batch.step(2)
    assert b.get_timing()["sweep_k"][1] > 0 and b.get_timing()["cfl"][1] == 2
    same(a, b, name)
    same(a, c, name)
    batch.set([])
    batch.close()
    for mm in (a, b, c):
        mm.close()


@pytest.mark.parametrize("threads", [64, 128, 192, 256])
@pytest.mark.parametrize("name", ["t2d", "t3dppm", "uppm"])
def test_tiles_read_back_can_be_set(name, threads):
    """The tiles a model reports are ones another model of its shape takes,
    and then has in use (a plan kept from an autotuned model)."""
    p = configs.ALL[name].resolved()
    g = native.setup_grid(p)
    m = native.setup_metric(p, g)
    a, b = native.Model(p, g, m), native.Model(p, g, m)
    a.set_block_sizes([threads] * len(native.TUNE_SLOTS))
    for seg in (0, 2, 64):
        a.set_sweep_tiles(0, seg, seg)
        plan = {**a.block_sizes(), **a.sweep_tiles()}
        b.set_block_sizes(plan)
        assert {**b.block_sizes(), **b.sweep_tiles()} == plan, seg
    a.close()
    b.close()
