"""Both forms of the rebuild stage where each changes shape.  The several
launches serve boxes of more than 256 x 256 cell columns, more than 262144
bonds, and lists of more than 16 entries a bond above 40960 bonds (160 below);
the one launch serves the rest.  Lists are checked against the cells' members
found on the host; failures inside a run against runs that meet none."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.helpers import uneven_system
from tests.scenarios import make_filaments
from tests.test_gpu_commit import _state
from tests.test_gpu_rebuild_edges import _cell_pairs, _spread, _system

pytestmark = pytest.mark.gpu


def _check(s, n1d, fil):
    assert s.counters()["n_cells_1d"] == n1d
    a, b = s.candidates()
    code = np.sort(np.minimum(a, b).astype(np.int64) * fil.nb + np.maximum(a, b))
    want = _cell_pairs(s.cell_keys().astype(np.int64), n1d, np.asarray(fil.site_off))
    np.testing.assert_array_equal(code, want)


def _fill(n1d, nb, part=1.0, delta=1e-4):
    """Two-bond filaments anywhere in the middle `part` of a box of n1d cells
    of side 2."""
    rng = np.random.default_rng(n1d + nb)
    p = sc.params_init(float(n1d), delta=delta, min_cell_length=2.0, seed=11)
    p.f_cutoff = 10.0
    u = rng.normal(size=(nb // 2, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    x = rng.uniform(-n1d, n1d, u.shape) * part
    sites = [a + np.arange(-1, 2)[:, None] * b for a, b in zip(x, u)]
    if nb % 2:
        sites[-1] = np.vstack([sites[-1], 2 * sites[-1][-1] - sites[-1][-2]])
    return p, make_filaments(sites)


# several launches: bonds at the edges of the list pass's groups of 256 and
# blocks of four groups
@pytest.mark.parametrize("nb", [255, 256, 257, 511, 513, 1023, 1024, 1025, 2047, 2049, 8191, 8192,
                                8193, 33000])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_bonds_of_the_several_launches(nb, precision):
    p, fil = _system(257, nb, nb)
    s = sc.FilamentSystem(p, fil, precision=precision, use_graph=True)
    _check(s, 257, fil)
    s.step(4)
    s.close()


# several launches because of long lists: columns at the edges of a scan tile
# of 4096, one tile and several; the lists of a rebuild inside a run, after the
# load's in one launch
@pytest.mark.parametrize("n1d", [63, 64, 65, 90, 91, 150, 256])
def test_columns_of_the_several_launches(n1d):
    p, fil = _fill(n1d, 41200, part=25.0 / n1d)
    s = sc.FilamentSystem(p, fil, precision="mixed", use_graph=True)
    assert 2 * s.counters()["n_candidates"] > 16 * fil.nb
    for steps in (0, 21, 20):
        s.step(steps)
        _check(s, n1d, fil)
    assert s.counters()["n_rebuilds"] > 1
    s.close()


# one launch: columns at the edges of a scan tile (2048 in blocks of 512
# threads, 4096 in blocks of 1024), many tiles, and the last box that it serves
@pytest.mark.parametrize("n1d, nb", [(45, 301), (46, 301), (64, 700), (65, 701), (90, 2000),
                                     (181, 400), (255, 300), (256, 300), (256, 5001), (63, 41201),
                                     (64, 41200), (65, 41201), (91, 41201), (150, 50001),
                                     (256, 60001)])
def test_columns_of_the_one_launch(n1d, nb):
    p, fil = _fill(n1d, nb, delta=1e-3)
    assert fil.nb == nb
    s = sc.FilamentSystem(p, fil, precision="fp64", use_graph=True)
    for steps in (0, 41):
        s.step(steps)
        _check(s, n1d, fil)
    assert s.counters()["n_rebuilds"] > 1
    s.close()


# several launches of large systems: several scan tiles and many groups
@pytest.mark.parametrize("n1d, nb", [(64, 262147), (91, 262400), (150, 300001)])
def test_large_systems(n1d, nb):
    p, fil = _fill(n1d, nb, delta=1e-3)
    s = sc.FilamentSystem(p, fil, precision="mixed", use_graph=True, spatial_order=True)
    for steps in (0, 41):
        s.step(steps)
        _check(s, n1d, fil)
    assert s.counters()["n_rebuilds"] > 1
    s.close()


@pytest.mark.parametrize("other", ["small", "crowded"])
def test_batch_in_several_launches(other):
    """A member of more than 262144 bonds beside a small one or one with long
    lists, no column scan in two launches: each as when stepped alone."""
    p, fil, _ = _spread(262400)
    cases = [(p, fil), _spread(700)[:2] if other == "small" else _fill(25, 9000, 0.5, 1e-3)]
    ens = sc.Ensemble(hbm_budget=8 << 30, max_active=4, steps_per_launch=16, batch_size=4)
    ids = [ens.submit(p, f, 41, precision="mixed") for p, f in cases]
    ens.drain(60)
    for i, (p, f) in zip(ids, cases):
        s = sc.FilamentSystem(p, f, precision="mixed", use_graph=True)
        s.step(41)
        assert s.counters()["n_rebuilds"] > 1
        np.testing.assert_array_equal(ens.result(i), s.sites()[0])
        s.close()
    ens.close()


def test_batch_replays_by_the_members_lists():
    """Two memberships that agree in sizes but whose rebuilds take the one and
    the several launches."""
    cases = [_fill(45, 41200, 1.0, 1e-3), _fill(45, 41200, 0.6, 1e-3)]
    mean = []
    ens = sc.Ensemble(hbm_budget=8 << 30, max_active=1, steps_per_launch=16, batch_size=4)
    for p, f in cases:
        rid = ens.submit(p, f, 42, precision="mixed")
        ens.drain(60)
        s = sc.FilamentSystem(p, f, precision="mixed", use_graph=True)
        mean.append(2 * s.counters()["n_candidates"] / f.nb)
        s.step(42)
        assert s.counters()["n_rebuilds"] > 1
        np.testing.assert_array_equal(ens.result(rid), s.sites()[0])
        s.close()
    assert mean[0] < 16 < mean[1]
    ens.close()


def _sparse():
    return uneven_system(copies=12, radius=150.0, delta=2e-4)


@pytest.mark.parametrize("graph", [False, True])
def test_capacity_growth_inside_a_run(graph):
    p, fil = _sparse()
    ref = sc.FilamentSystem(p, fil, precision="mixed", use_graph=graph)
    assert ref.counters()["n_cells_1d"] > 256
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


@pytest.mark.parametrize("graph", [False, True])
def test_unphysical_step_inside_a_run(graph):
    seen = []
    for delta in (5e-3, 2e-2, 1e-1):
        p, fil = _sparse()
        p.delta = delta
        at = []
        for n in (1, 64):
            s = sc.FilamentSystem(p, fil, precision="fp64", use_graph=graph)
            assert s.counters()["n_cells_1d"] > 256
            with pytest.raises(sc.UnphysicalResult):
                for _ in range(640 // n):
                    s.step(n)
            at.append(s.counters()["i_step"])
            s.close()
        assert at[0] == at[1]
        seen.append(at[0])
    assert any(2 < k < 64 for k in seen), seen
