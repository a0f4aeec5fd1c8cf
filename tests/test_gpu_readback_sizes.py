"""Read-back on both sides of the sizes from which a kernel puts an array into
the caller's order and precision: 49152 FP64 and 196608 FP32 values in spatial
order, 2^20 FP32 values in the caller's; and of the size (16384 values) up to
which both statistics come in one copy."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.scenarios import make_filaments

pytestmark = pytest.mark.gpu


def _lattice(ns, sites=32):
    """Straight filaments along z on a lattice too wide for pairs, ns sites in
    all, in random order."""
    nf = ns // sites
    lengths = np.full(nf, sites)
    lengths[: ns - nf * sites] += 1
    side = int(np.ceil(nf ** 0.5))
    spots = np.random.default_rng(ns).permutation(side * side)[:nf]
    x = 4.0 * (np.stack([spots // side, spots % side], axis=1) - 0.5 * side)
    fil = [np.concatenate([np.tile(a, (n, 1)), np.arange(n)[:, None] - 0.5 * n], axis=1)
           for a, n in zip(x, lengths)]
    p = sc.params_init(max(40.0, 2.0 * side + 4.0), delta=1e-5, min_cell_length=8.0, seed=5)
    return p, make_filaments(fil)


@pytest.mark.parametrize("precision, ns", [("fp64", 16383), ("fp64", 16384), ("mixed", 16385),
                                           ("mixed", 65535), ("mixed", 65536), ("fp64", 50000),
                                           ("mixed", 349525), ("mixed", 349526)])
def test_arrays_in_either_storage_order(precision, ns):
    p, fil = _lattice(ns)
    assert fil.ns == ns
    a = sc.FilamentSystem(p, fil, precision=precision, spatial_order=True)
    b = sc.FilamentSystem(p, fil, precision=precision, spatial_order=False)
    np.testing.assert_array_equal(a.sites()[0], fil.r)
    for s in (a, b):
        s.step(2)
    force = a.sites()[2]
    assert np.count_nonzero(force) > 0.9 * force.size
    for x, y in zip(a.sites() + (a.tensions(), a.dr_state()),
                    b.sites() + (b.tensions(), b.dr_state())):
        np.testing.assert_array_equal(x, y)
    a.close()
    b.close()


@pytest.mark.parametrize("nf", [1, 5461, 5462, 20000])
def test_statistics(nf):
    p, fil = _lattice(3 * nf, sites=3)
    s = sc.FilamentSystem(p, fil, precision="mixed", spatial_order=True)
    x, off = fil.r.reshape(3, -1), fil.site_off
    e2e, com = s.filament_stats()
    np.testing.assert_array_equal(e2e, x[:, off[1:] - 1] - x[:, off[:-1]])
    want = np.add.reduceat(x, off[:-1], axis=1) / 3
    np.testing.assert_allclose(com, want, rtol=0, atol=3 * 2.0 ** -52 * np.abs(x).max())
    s.close()
