"""The compact metric tables (an axisymmetric metric that couples theta to
nothing: 13 planes a kernel reads, derived values among them) against the
general ones: the same model with a zero of the centre metric negated, which
keeps every value but not the structure the compact form asks for bit by
bit.  State, time, counters and stored fluxes bit for bit, for every
reconstruction, wave-speed formula, recovery and precision."""
import numpy as np
import pytest

from raishinsource_amd import configs, native
from test_gpu_tiles import same

pytestmark = pytest.mark.gpu


def make(p, general, mixed):
    p = p.resolved()
    g = native.setup_grid(p)
    m = native.setup_metric(p, g)
    uri = (native.setup_tube(p, *native.random_tube_states(np.random.default_rng(3))) if p.model == 2
           else native.setup_torus(p, g, m, seed=1))
    if general:
        m["gcov"][0, 3] = -0.0
    mod = native.Model(p, g, m)
    mod.set_state(uri)
    mod.set_precision(mixed)
    return mod


@pytest.mark.parametrize("name,mixed,steps", [
    ("uppm", False, 3), ("uppm", True, 3), ("t2d", False, 3), ("t2dgam", False, 2), ("t2drc2", False, 2),
    ("umc", False, 3), ("uleis", False, 3), ("urc2", True, 3), ("ump5", False, 1), ("uweno", True, 1),
    ("utube", False, 4)])
def test_compact_tables_equal_general(name, mixed, steps):
    a, b = make(configs.ALL[name], False, mixed), make(configs.ALL[name], True, mixed)
    for q in range(4):
        assert np.array_equal(a.tables(q), b.tables(q)), q
    assert a.cdtcfl4() == b.cdtcfl4()
    for s in range(steps):
        assert np.array_equal(a.step(1), b.step(1), equal_nan=True), s
    same(a, b, name)
    a.close()
    b.close()
