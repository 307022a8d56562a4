"""Reading small buffers through one pinned copy (kg_read_agents,
kg_ensemble_read) on both sides of the size where reads turn to plain
copies, and partial, empty and refused reads."""
import ctypes

import numpy as np
import pytest

from krabmaga_amd import Ensemble, Field2D, FlockParams, KgError, RunSpec, _abi

pytestmark = pytest.mark.gpu

D = 10.0 / 1.5


@pytest.mark.parametrize("n", [1, 255, 257, 32767, 32768, 32769, 50000])
def test_read_returns_what_was_set(n):
    rng = np.random.default_rng(n)
    side = 2000.0
    a = {"id": rng.permutation(n).astype(np.uint32)}
    for k in ("x", "y", "hx", "hy"):
        a[k] = (rng.random(n) * side).astype(np.float32)
    f = Field2D(side, side, D, True, n + 3)
    f.set_object_locations(a["id"], a["x"], a["y"], a["hx"], a["hy"])
    w = f.read_agents(1)  # insertion order
    f.lazy_update()
    r = f.read_agents(0)
    assert len(f.read_agents(1)["id"]) == 0
    for k in a:
        assert np.array_equal(w[k], a[k]), k
        assert len(r[k]) == n
    o = np.argsort(r["id"])
    for k in ("x", "y", "hx", "hy"):
        assert np.array_equal(r[k][o], a[k][np.argsort(a["id"])]), k
    # some arrays only, and a buffer too small
    L, m = _abi.lib(), ctypes.c_size_t()
    x = np.zeros(n, np.float32)
    assert L.kg_read_agents(f._h, 0, None, _abi.f32p(x), None, None, None, n, ctypes.byref(m)) == 0
    assert m.value == n and np.array_equal(x, r["x"])
    rc = L.kg_read_agents(f._h, 0, None, _abi.f32p(x), None, None, None, n - 1, ctypes.byref(m))
    assert rc == _abi.KG_E_CAPACITY and m.value == n
    f.close()


def test_read_reports_a_location_outside_the_grid():
    # y wraps by the width: on a field wider than tall a bird can leave it
    f = Field2D(400.0, 100.0, D, True, 2)
    f.set_object_locations([0], [50.0], [99.9], [0.0], [1.0])
    f.schedule_run(FlockParams(momentum=1.0, randomness=0.0, jump=30.0), 0, 1)
    with pytest.raises(KgError):
        f.read_agents(0)
    f.close()


@pytest.mark.parametrize("path", [{}, {"tile_resident": True}, {"binned": True}])
def test_ensemble_reads_small_and_large_runs(path):
    specs = [RunSpec(width=float(np.sqrt(n / 0.025)), height=float(np.sqrt(n / 0.025)), agents=n,
                     params=FlockParams(seed=n), init_seed=n) for n in (1, 900, 32768, 32769)]
    with Ensemble() as ens:
        ids = ens.admit(specs)
        ens.run(3, **path)
        for rid, s in zip(ids, specs):
            st, i = ens.state_by_id(rid)
            f = Field2D(s.width, s.height, s.discretization, True, s.agents)
            f.init_uniform(s.agents, s.init_seed, s.heading_mode)
            f.schedule_run(s.params, 0, 3)
            ref, _ = f.state_by_id(0)
            f.close()
            assert np.array_equal(i, np.arange(s.agents))
            assert np.array_equal(st.view(np.uint32), ref.view(np.uint32))
