"""cdtcfl4 (cdtcfl.f90:2) where a workgroup of the reduction takes more than
one 256-cell chunk: the reference's running MIN (a NaN element restarts it)
against the oracle, bit for bit, with NaN cells at the start, inside and at
the end of chunks and workgroups, and as the last cell of all."""
import ctypes as C
from dataclasses import replace

import numpy as np
import pytest

from harness import Oracle, synthetic_state
from raishinsource_amd import configs, native
from test_gpu_tiles import bitdiff

pytestmark = pytest.mark.gpu

P = replace(configs.U_PPM, name="cfl", imax=80, jmax=72, kmax=66).resolved()
NC = (P.imax - 2) * (P.jmax - 2) * (P.kmax - 2)  # 1365 chunks and a remainder: two chunks a workgroup


@pytest.fixture(scope="module")
def setup(oracle_lib):
    g = native.setup_grid(P)
    m = native.setup_metric(P, g)
    mod = native.Model(P, g, m)
    yield g, m, synthetic_state(P, seed=4), mod
    mod.close()


@pytest.mark.parametrize("cells", [[], [0], [255], [256, 511, 512], [300, 900, 100000], [NC - 2], [NC - 1],
                                   list(range(512, 1024)), list(range(NC - 300, NC))])
def test_nan_cells(setup, cells):
    g, m, uri, mod = setup
    w = uri.copy(order="F")
    ci, cj = P.imax - 2, P.jmax - 2
    for q, t in enumerate(cells):  # position t of the box in (k, j, i) order
        w[(0, 1, 4)[q % 3], 1 + t % ci, 1 + (t // ci) % cj, 1 + t // (ci * cj)] = np.nan
    d = [C.c_double(0) for _ in range(4)]
    Oracle(P).call("cdtcfl4", w, m["gcov"], m["gcon"], C.byref(d[0]), g["dx1b"], g["dx2b"], g["dx3b"], C.byref(d[1]),
                   C.byref(d[2]), C.byref(d[3]), P.nm1)
    mod.set_state(w)
    want = np.array([x.value for x in d])
    got = np.array(mod.cdtcfl4())
    assert bitdiff(got, want) == 0, (got, want)
