"""The gather rebinning's slow way (a tile of more candidates than its
work-group holds, a bin past 512 birds, past 2,048, an overflowed outbox, birds
from further than the neighbouring tiles) and
the fields it leaves to the scatter (not square, jumps past a tile): after
every step the read buffer equals the oracle's, bit for bit."""
import numpy as np
import pytest

from krabmaga_amd import Field2D, FlockParams

pytestmark = pytest.mark.gpu

D = 10.0 / 1.5


def crowds(rng, width, height, spread, sizes):
    """Uniform birds and crowds, each within one cell."""
    xs, ys = [rng.uniform(0.0, width, spread)], [rng.uniform(0.0, height, spread)]
    for m in sizes:
        cx, cy = rng.integers(0, int(width / D) - 1), rng.integers(0, int(height / D) - 1)
        xs.append((cx + rng.uniform(0.05, 0.95, m)) * D)
        ys.append((cy + rng.uniform(0.05, 0.95, m)) * D)
    x = np.concatenate(xs).astype(np.float32)
    y = np.concatenate(ys).astype(np.float32)
    a = rng.uniform(0.0, 2.0 * np.pi, x.size)
    return x, y, np.cos(a).astype(np.float32), np.sin(a).astype(np.float32)


@pytest.mark.parametrize("width,height,jump,spread,sizes", [
    (600.0, 600.0, 0.05, 5000, (2049, 513, 257, 65, 9)),  # bins at the sorts' edges
    (600.0, 600.0, 0.7, 8000, (300,) * 12),               # tiles past 2,048 birds
    (400.0, 400.0, 80.0, 6000, ()),                       # outboxes past 256 birds
    (500.0, 500.0, 400.0, 4000, ()),                      # jumps past a tile: scattered
    (300.0, 700.0, 0.7, 4000, (700,)),                    # y wraps by the width: scattered
])
def test_every_rebinning_equals_the_oracle(oracle, width, height, jump, spread, sizes):
    rng = np.random.default_rng(spread)
    x, y, hx, hy = crowds(rng, width, height, spread, sizes)
    n, steps = x.size, 3
    p = FlockParams(seed=7, jump=jump)
    f = Field2D(width, height, D, True, n)
    f.set_object_locations(np.arange(n, dtype=np.uint32), x, y, hx, hy)
    f.lazy_update()
    for s in range(steps):
        f.flock_step(p, s)
        f.lazy_update()
    got, ids = f.state_by_id(0)
    fl = oracle.Flocker(width, height, D, True, x, y, hx, hy, oracle.params(seed=7, jump=jump))
    fl.step(steps)
    assert np.array_equal(ids, np.arange(n))
    assert np.array_equal(got.view(np.uint32), fl.state().view(np.uint32))


def test_birds_without_a_position_go_to_the_first_cell(oracle):
    """An infinite heading makes a position NaN, which lies in cell 0 of its
    axis: the gather finds such birds though they pass many tiles."""
    rng = np.random.default_rng(3)
    x, y, hx, hy = crowds(rng, 700.0, 700.0, 9000, ())
    far = np.flatnonzero((x > 300.0) & (y > 300.0))[:4]
    hx[far[:2]] = np.inf
    hy[far[1:]] = -np.inf
    n, steps = x.size, 3
    p = FlockParams(seed=7)
    f = Field2D(700.0, 700.0, D, True, n)
    f.set_object_locations(np.arange(n, dtype=np.uint32), x, y, hx, hy)
    f.lazy_update()
    for s in range(steps):
        f.flock_step(p, s)
        f.lazy_update()
    got, ids = f.state_by_id(0)
    fl = oracle.Flocker(700.0, 700.0, D, True, x, y, hx, hy, oracle.params(seed=7))
    fl.step(steps)
    want = fl.state()
    assert np.array_equal(ids, np.arange(n)) and np.isnan(want).any()
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all()
