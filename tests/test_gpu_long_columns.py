"""Candidate lists with long cell columns: numbers of bonds in a column at the
edges of what 16 lanes sort (96), of a lane's bonds in a round of a long column
(256) and of a wavefront's stage (384), beside short and empty columns, in the
one-launch rebuild and in the several launches."""
import numpy as np
import pytest

import simcore_amd as sc
from oracle.oracle_py import OracleSystem
from tests.scenarios import make_filaments
from tests.test_gpu_rebuild_edges import _cell_pairs

pytestmark = pytest.mark.gpu


def _columns(n1d, population, seed):
    """Filaments of two bonds along z, `population[x, y]` bonds in all in cell
    column (x, y) of a box of n1d cells of side 2."""
    rng = np.random.default_rng(seed)
    col = np.repeat(np.arange(n1d * n1d), np.ravel(population) // 2)
    c = np.stack([col // n1d, col % n1d], axis=1)
    xy = 2.0 * (c + rng.uniform(0.1, 0.9, c.shape)) - n1d
    z = rng.uniform(-n1d, n1d, len(col))
    start = np.concatenate([xy, z[:, None]], axis=1)
    order = rng.permutation(len(col))
    p = sc.params_init(float(n1d), delta=1e-6, min_cell_length=2.0, seed=11)
    step = np.array([0.0, 0.0, 1.0])
    return p, make_filaments([x + np.arange(3)[:, None] * step for x in start[order]])


def _check(p, fil, n1d, population, precision):
    s = sc.FilamentSystem(p, fil, precision=precision, use_graph=True)
    keys = s.cell_keys().astype(np.int64)
    np.testing.assert_array_equal(np.bincount(keys // n1d, minlength=n1d * n1d),
                                  np.ravel(population))
    a, b = s.candidates()
    code = np.sort(np.minimum(a, b).astype(np.int64) * fil.nb + np.maximum(a, b))
    np.testing.assert_array_equal(code, _cell_pairs(keys, n1d, np.asarray(fil.site_off)))
    return s


@pytest.mark.parametrize("where, bonds", [("one", n) for n in (94, 96, 98, 254, 256, 258, 384, 386,
                                                               770, 1500)] +
                         [("some", n) for n in (96, 98, 258, 382, 386, 640)] +
                         [("all", n) for n in (96, 98)])
def test_lists_of_long_columns(where, bonds):
    n1d = 11  # 121 columns: the last wavefront has one
    rng = np.random.default_rng(bonds)
    population = 2 * rng.integers(0, 8, (n1d, n1d))
    if where == "one":
        population[n1d - 1, n1d - 1] = bonds
    elif where == "some":
        population[rng.random((n1d, n1d)) < 0.1] = bonds
    else:
        population[:] = bonds - 2 * rng.integers(0, 2, (n1d, n1d))
    p, fil = _columns(n1d, population, bonds)
    s = _check(p, fil, n1d, population, "fp64")
    if where == "one":  # the order of each list, by the sums it gives
        ora = OracleSystem(p, fil)
        s.step(2)
        assert ora.step(2) == 0
        for x, y in zip(s.bond_forces(), ora.bond_forces()):
            np.testing.assert_array_equal(x, y)
        ora.close()
    s.close()


def test_lists_of_long_columns_in_several_launches():
    n1d = 64
    rng = np.random.default_rng(3)
    population = 2 * rng.integers(0, 62, (n1d, n1d))
    population[rng.random((n1d, n1d)) < 0.02] = 386
    population[5:9, 20:24] = 900
    p, fil = _columns(n1d, population, 3)
    assert fil.nb > 262144
    _check(p, fil, n1d, population, "mixed").close()
