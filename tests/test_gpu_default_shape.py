"""A handle whose caller chose no launch shape: it says the balanced pair kernel
(0) however long its lists are, and its results, of whichever kernel it takes by
their length, are those of either kernel chosen by the caller, at load and after
a restored state."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.scenarios import make_filaments
from tests.test_gpu_pair_split import _system as split_system

pytestmark = pytest.mark.gpu


def _system(nb, n1d, spread=1.0, seed=3):
    """Filaments of two bonds in a box of n1d cells of side 2, in its middle
    `spread` part."""
    rng = np.random.default_rng(seed)
    p = sc.params_init(float(n1d), delta=1e-5, min_cell_length=2.0, seed=11)
    p.f_cutoff = 10.0
    u = rng.normal(size=(nb // 2, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    x = rng.uniform(-n1d, n1d, u.shape) * spread
    return p, make_filaments([a + np.arange(-1, 2)[:, None] * b for a, b in zip(x, u)])


def _mean(s):
    return 2.0 * s.counters()["n_candidates"] / s.nb


@pytest.mark.parametrize("nb, n1d, balanced", [(4000, 10, True), (8000, 10, False),
                                               (40000, 30, True), (40000, 20, False),
                                               (70000, 44, True), (70000, 36, False),
                                               (140000, 64, True), (140000, 52, False),
                                               (200000, 52, True)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_by_the_length_of_the_lists(nb, n1d, balanced, precision):
    p, fil = _system(nb, n1d)
    s = sc.FilamentSystem(p, fil, precision=precision, use_graph=True)
    line = next(x for n, x in ((32768, 160), (65536, 80), (131072, 32), (199999, 16), (1e9, 40))
                if nb <= n)
    assert (_mean(s) <= line) == balanced
    start = s.launch_shape()
    assert start["pair_block"] == 0
    s.step(6)
    assert s.launch_shape() == start
    for block in (0, 128):
        t = sc.FilamentSystem(p, fil, precision=precision, use_graph=True)
        shape = dict(start, pair_block=block)
        t.set_launch_shape(**shape)
        t.step(6)
        assert t.launch_shape() == shape  # the caller's choice stays
        for x, y in zip(s.sites() + s.bond_forces(), t.sites() + t.bond_forces()):
            np.testing.assert_array_equal(x, y)
        t.close()
    s.close()


def test_follows_a_restored_state():
    p, crowded = _system(8000, 20, spread=0.4)
    _, sparse = _system(8000, 20)
    a = sc.FilamentSystem(p, crowded, precision="mixed", use_graph=True)
    b = sc.FilamentSystem(p, sparse, precision="mixed", use_graph=True)
    assert _mean(a) > 160 > _mean(b)
    early, late = b.checkpoint(), a.checkpoint()
    b.step(4)
    ref = b.sites()[0]
    b.restore(late)
    a.step(4)
    b.step(4)
    assert a.launch_shape()["pair_block"] == b.launch_shape()["pair_block"] == 0
    np.testing.assert_array_equal(a.sites()[0], b.sites()[0])
    b.restore(early)
    b.step(4)
    np.testing.assert_array_equal(b.sites()[0], ref)
    a.close()
    b.close()


# the balanced kernel where the lists are too long for it to be the library's
# choice, at the edges of the rule of its bonds per wavefront
@pytest.mark.parametrize("thermo", [False, True])
@pytest.mark.parametrize("nb, precision", [(65536, "mixed"), (65537, "fp64"), (131072, "mixed"),
                                           (131073, "mixed"), (131073, "fp64")])
def test_balanced_kernel_by_choice_on_long_lists(nb, precision, thermo):
    a, b = split_system(nb, precision, thermo), split_system(nb, precision, thermo)
    assert _mean(a) > 80
    start = a.launch_shape()
    a.set_launch_shape(**start)
    b.set_launch_shape(**dict(start, pair_block=128))
    a.step(6)
    b.step(6)
    for x, y in zip(a.sites() + a.bond_forces(), b.sites() + b.bond_forces()):
        np.testing.assert_array_equal(x, y)
    if thermo:
        np.testing.assert_array_equal(a.bond_energies(), b.bond_energies())
        # (tolerance as where this system comes from)
        pa, pb = a.calculate_pressure(6), b.calculate_pressure(6)
        tol = 3 * nb * 2.0 ** -53 * max(1.0, np.abs(pb["pressure_tensor"]).max())
        np.testing.assert_allclose(pa["pressure_tensor"], pb["pressure_tensor"], rtol=0, atol=tol)
    a.close()
    b.close()
