"""Runs of steps that commit once per run against the same steps taken one by
one: counters, displacement bookkeeping, and the step an unphysical
displacement or a full candidate list is met at."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.helpers import c0_system, uneven_system

pytestmark = pytest.mark.gpu

RUNS = [1, 2, 3, 8, 9, 10, 16, 17, 27, 64]  # single steps, pairs, graphs of four pairs


def _state(s):
    c = s.counters()
    return [np.array(list(c.values())), s.dr_state(), s.tensions(), *s.sites(), *s.bond_forces()]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("graph", [False, True])
def test_runs_equal_single_steps(precision, graph):
    p, fil = uneven_system()
    one = sc.FilamentSystem(p, fil, precision=precision, use_graph=graph)
    run = sc.FilamentSystem(p, fil, precision=precision, use_graph=graph)
    for n in RUNS:
        for _ in range(n):
            one.step(1)
        run.step(n)
        for a, b in zip(_state(one), _state(run)):
            np.testing.assert_array_equal(a, b)
    assert run.counters()["n_rebuilds"] > 3
    one.close()
    run.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("graph", [False, True])
def test_unphysical_step_is_the_same_in_a_run(precision, graph):
    seen = []
    for delta in (2e-3, 3e-3, 1e-2):
        p, fil = c0_system()
        p.delta = delta
        at = []
        for n in (1, 64):
            s = sc.FilamentSystem(p, fil, precision=precision, use_graph=graph)
            with pytest.raises(sc.UnphysicalResult):
                for _ in range(400 // n):
                    s.step(n)
            at.append(s.counters()["i_step"])
            s.close()
        assert at[0] == at[1]
        seen.append(at[0])
    # met inside a run, where no commit launch precedes the odd step
    assert any(2 < k < 64 for k in seen), seen


@pytest.mark.parametrize("graph", [False, True])
def test_capacity_growth_inside_a_run(graph):
    p, fil = uneven_system(phi=0.08)
    ref = sc.FilamentSystem(p, fil, precision="mixed", use_graph=graph)
    n0 = ref.counters()["n_candidates"]
    s = sc.FilamentSystem(p, fil, precision="mixed", use_graph=graph, capacity_factor=-float(n0))
    b0 = s.device_bytes()
    for q in (ref, s):
        q.step(301)
    assert s.device_bytes() > b0
    for a, b in zip(_state(ref), _state(s)):
        np.testing.assert_array_equal(a, b)
    ref.close()
    s.close()
