"""A field filled anew with more and with fewer birds, run with graphs and the
same parameters each time: every run equals one on a new field, bit for bit.
The steps are captured once per population where their launches hold its
count."""
import numpy as np
import pytest

from krabmaga_amd import Field2D, FlockParams

pytestmark = pytest.mark.gpu

D = 10.0 / 1.5
SIDE = 600.0


def _birds(n, crowd, seed):
    """`crowd` of n birds round one spot, the others uniform."""
    rng = np.random.default_rng(seed)
    x, y = rng.uniform(0.0, SIDE, (2, n))
    x[:crowd] = 300.0 + rng.normal(0.0, 8.0, crowd)
    y[:crowd] = 300.0 + rng.normal(0.0, 8.0, crowd)
    a = rng.uniform(0.0, 2.0 * np.pi, n)
    return [np.arange(n, dtype=np.uint32)] + [v.astype(np.float32)
                                              for v in (x, y, np.cos(a), np.sin(a))]


@pytest.mark.parametrize("jump,crowd", [
    (0.7, 9000),   # crowded tiles: birds stepped by runs of the read buffer
    (60.0, 0),     # jumps past a tile: rebinned by scatter
    (0.7, 0),      # two launches a step, whose graphs serve every population
])
def test_each_population_equals_a_new_field(jump, crowd):
    p = FlockParams(seed=5, jump=jump)
    counts = (14000, 17000, 11000, 14000)
    f = Field2D(SIDE, SIDE, D, True, max(counts))
    for k, (n, steps) in enumerate([(n, s) for n in counts for s in (7, 8)]):
        birds = _birds(n, crowd, k)
        f.set_object_locations(*birds)
        f.schedule_run(p, 0, steps)
        got, ids = f.state_by_id(0)
        g = Field2D(SIDE, SIDE, D, True, max(counts))
        g.set_object_locations(*birds)
        g.schedule_run(p, 0, steps, use_graph=False)
        ref, rids = g.state_by_id(0)
        g.close()
        assert np.array_equal(ids, rids)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (n, steps)
