"""The forms a model's step takes (launches shared or apart, one kernel or
two, the tiles and sizes in use) as a caller meets them: which models make a
batch, what the timers and getters report."""
from dataclasses import replace

import pytest

from raishinsource_amd import configs, native
from test_gpu_tiles import make, same

pytestmark = pytest.mark.gpu


def test_batch_of_mc_and_split_ppm():
    """MC models and PPM models of the split form make one batch (their steps
    are the same sequence of launches); MC and WENO5 do not."""
    ps = [configs.U_MC, configs.U_PPM, replace(configs.T2D_MC, name="t2dmc_b", icha=1), configs.T2D]
    alone = [make(p, q == 2, seed=q) for q, p in enumerate(ps)]
    batched = [make(p, q == 2, seed=q) for q, p in enumerate(ps)]
    for mm in alone + batched:
        if mm.p.irec == 5:
            mm.set_sweep_tiles(1, 0, 0)
    for mm in alone:
        mm.step(4)
    b = native.Batch(batched)
    b.step(1)
    b.step_graph(1)
    b.step(1)
    for x, y in zip(alone, batched):
        same(x, y, x.p.name)
    w = make(replace(configs.U_WENO, irkt=2))
    with pytest.raises(native.RaishinError, match="different step sequences"):
        b.set([batched[0], w])
    b.set([])
    b.close()
    for mm in alone + batched + [w]:
        mm.close()


@pytest.mark.parametrize("threads", [64, 128, 256])
@pytest.mark.parametrize("ni,nj,nk", [(40, 24, 40), (64, 64, 64), (251, 57, 77)])
def test_untuned_tiles_are_ones_the_autotuner_times(ni, nj, nk, threads):
    """A tile is its cells along the axis (a workgroup's), in the rule as in
    what can be asked for, so tuning can keep what an untuned model has."""
    p = configs.Pram("tile", ni, nj, nk, irec=5, irkt=3).resolved()
    m = native.Model.from_grid(p, native.setup_grid(p))
    m.set_block_sizes([threads] * 8)
    for seg in m.sweep_tiles()["seg_j"], m.sweep_tiles()["seg_k"]:
        assert seg in (8, 16, 32, 64)
    m.close()


@pytest.mark.parametrize("threads,seg", [(256, 4), (256, 2), (192, 4), (128, 2), (64, 64), (192, 64)])
def test_smallest_and_tallest_tiles_equal_split(threads, seg):
    p = configs.Pram("tile", 75, 17, 71, irec=5, irkt=3, cfl=0.4)
    a, b = make(p), make(p)
    a.set_sweep_tiles(1, 0, 0)
    b.set_block_sizes([threads] * 8)
    b.set_sweep_tiles(0, seg, seg)
    for s in range(2):
        assert a.step(1) == b.step(1), s
    same(a, b, threads)
    a.close()
    b.close()


def general_metric(p, table="gcov", mixed=False, seed=1):
    """A model whose metric has not the compact tables' structure, or whose
    Christoffel tables are not symmetric: a zero of one table negated, which
    keeps every value."""
    p = p.resolved()
    g = native.setup_grid(p)
    m = native.setup_metric(p, g)
    uri = native.setup_torus(p, g, m, seed=seed, noise=0.02)
    at = (0, 3) if table == "gcov" else (3, 2, 3)
    assert not m[table][at].any()
    m[table][at] = -0.0
    mod = native.Model(p, g, m)
    mod.set_state(uri)
    mod.set_precision(mixed)
    return mod


def test_sizes_and_tiles_reported_are_those_in_use():
    """Sweeps that share a launch have one workgroup size, sweep i's: the
    sizes read back say so, and the tiles are those of that size."""
    odd = [256, 64, 192, 128, 64, 192, 128, 64]
    a, b = make(configs.T3D_PPM), make(configs.T3D_PPM)
    a.set_block_sizes(odd)
    b.set_block_sizes([256, 64, 64, 64, 64, 192, 128, 64])
    assert a.block_sizes() == b.block_sizes()
    assert a.sweep_tiles() == b.sweep_tiles()
    a.set_sweep_tiles(1, 0, 0)  # the split form's sweeps are launches of their own
    assert list(a.block_sizes().values()) == odd
    a.close()
    b.close()
    c, d = make(configs.U_MP5), general_metric(configs.U_MP5)
    for mm, want in ((c, [64, 64, 64]), (d, [64, 192, 128])):
        mm.set_block_sizes(odd)
        assert [mm.block_sizes()[k] for k in ("sweep_i", "sweep_j", "sweep_k")] == want
        mm.close()


@pytest.mark.parametrize("table", ["gcov", "christ"])
def test_recovery_timed_where_it_is_a_kernel_of_its_own(table):
    """Kind 4 (update) and kind 9 (recov) of a model whose step makes a launch
    of each; the autotuner then has samples of both."""
    a, b = make(configs.U_PPM, seed=1), general_metric(configs.U_PPM, table)
    for mm, recov in ((a, 0), (b, 6)):
        mm.set_timing(True)
        mm.step(3)
        t = mm.get_timing()
        assert t["update"][1] == 6 and t["recov"][1] == recov, t
    same(a, b, table)
    a.close()
    b.close()


def test_general_tables_in_a_batch():
    """Members with general metric tables or asymmetric Christoffel tables (two
    kernels at the place of the others' one) beside one with neither."""
    members = [("gcov", False), ("christ", False), ("gcov", True), ("christ", True)]
    def build():
        return [general_metric(configs.U_PPM, t, mx, q) for q, (t, mx) in enumerate(members)] + [
            make(configs.T2D, seed=4), general_metric(replace(configs.T2D, name="t2d_rc2", iwvec=2), "gcov", False, 5)]
    alone, batched = build(), build()
    for mm in alone:
        mm.step(4)
    b = native.Batch(batched)
    b.step(1)
    b.step_graph(1)
    b.step(1)
    for q, (x, y) in enumerate(zip(alone, batched)):
        same(x, y, q)
    b.set([])
    b.close()
    for mm in alone + batched:
        mm.close()
