"""Ensembles that mix runs of many birds with runs of many bins: each fits the
resident step alone, together they may not fit one launch's LDS, and every run
still gives the bits it gives alone."""
import os
import subprocess

import numpy as np
import pytest

from krabmaga_amd import Ensemble, Field2D, FlockParams, RunSpec, Tuning

NEAR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "near")


def test_runs_of_one_launch_fit_its_lds():
    subprocess.run(["make", "-s", "-C", NEAR, os.path.join(NEAR, "group_check")], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    r = subprocess.run([os.path.join(NEAR, "group_check")], capture_output=True, text=True,
                       timeout=300, env=env)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "0 scenario(s) failed" in r.stdout


def _run(n, side, seed):
    return RunSpec(width=side, height=side, agents=n,
                   params=FlockParams(radius=10.0, seed=seed * 7919 + 3), init_seed=seed)


@pytest.mark.gpu
@pytest.mark.parametrize("tuning,other", [
    (Tuning(), (200, 27000.0)),                                   # 163,868 bytes together
    (Tuning(tile_cols=8, tile_rows=32, bin_rows=1), (500, 1000.0)),  # 195,612 bytes
    (Tuning(), (1000, 200.0)),                                    # one launch
])
def test_many_birds_beside_many_bins(tuning, other):
    specs = [_run(4096, 404.8, 1), _run(other[0], other[1], 2)]
    with Ensemble(tuning) as ens:
        ids = ens.admit(specs)
        ens.run(5)
        ens.run(7)
        got = [ens.state_by_id(i) for i in ids]
    for s, (state, order) in zip(specs, got):
        f = Field2D(s.width, s.height, s.discretization, True, s.agents)
        f.init_uniform(s.agents, s.init_seed, s.heading_mode)
        f.schedule_run(s.params, 0, 12)
        ref, rids = f.state_by_id(0)
        assert np.array_equal(order, rids)
        assert np.array_equal(state.view(np.uint32), ref.view(np.uint32))


@pytest.mark.gpu
def test_a_short_tail_is_not_rebuilt_for_the_resident_step():
    """When the last run past the resident step's size has retired, the layout
    is kept for a few steps more: a rebuild costs more than they do.  (The
    retired run is under a third of the tiles, so nothing else asks for one.)"""
    specs = [_run(900 + 100 * i, 250.0, 3 + i) for i in range(16)] + [_run(6000, 490.0, 20)]
    with Ensemble() as ens:
        ids = ens.admit(specs)
        ens.run(3)
        ens.retire(ids[-1])
        builds = ens.stats()["builds"]
        ens.run(1)
        ens.run(1)
        assert ens.stats()["builds"] == builds
        ens.run(40)
        ens.run(2)
        assert ens.stats()["builds"] == builds + 1
        got = [ens.state_by_id(i) for i in ids[:-1]]
    for s, (state, order) in zip(specs, got):
        f = Field2D(s.width, s.height, s.discretization, True, s.agents)
        f.init_uniform(s.agents, s.init_seed, s.heading_mode)
        f.schedule_run(s.params, 0, 47)
        ref, rids = f.state_by_id(0)
        assert np.array_equal(order, rids)
        assert np.array_equal(state.view(np.uint32), ref.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("before", [0, 5])
def test_a_build_that_fails_leaves_the_runs_to_the_next(before):
    """60,000 birds on 6 x 6 cells fit no LDS class of the tile-resident form:
    the run is refused again and again, and steps in the bin-grouped form as it
    would alone, with the run that was there before it."""
    small, dense = _run(5000, 450.0, 40), _run(60000, 40.0, 41)
    with Ensemble() as ens:
        ids = ens.admit([small])
        if before:
            ens.run(before, tile_resident=True)
        ids += ens.admit([dense])
        for _ in range(2):
            with pytest.raises(Exception, match="LDS budget"):
                ens.run(1, tile_resident=True)
        ens.run(2, binned=True)
        got = [ens.state_by_id(i) for i in ids]
        assert [ens.steps(i) for i in ids] == [before + 2, 2]
    for s, steps, (state, order) in zip((small, dense), (before + 2, 2), got):
        f = Field2D(s.width, s.height, s.discretization, True, s.agents)
        f.init_uniform(s.agents, s.init_seed, s.heading_mode)
        f.schedule_run(s.params, 0, steps)
        ref, rids = f.state_by_id(0)
        assert np.array_equal(order, rids)
        assert np.array_equal(state.view(np.uint32), ref.view(np.uint32))
