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
