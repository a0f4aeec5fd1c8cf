"""Read-back in the caller's order and the on-device analyses, at the sizes
where their code paths change: below and above the size from which a kernel
reorders, filaments of 3 to 256 sites, histogram shapes at the edge of the
block-local counters."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.scenarios import make_filaments

pytestmark = pytest.mark.gpu


def _straight(lengths, seed, box):
    """Straight random filaments, spread so thinly that none interact."""
    rng = np.random.default_rng(seed)
    out = []
    for n in lengths:
        u = rng.normal(size=3)
        u /= np.linalg.norm(u)
        out.append(rng.uniform(-0.5, 0.5, 3) * box + np.arange(n)[:, None] * u)
    return out


# 3 values per site, 16384 the size from which the device reorders
@pytest.mark.parametrize("ns_min", [30, 5300, 5600, 40000])
@pytest.mark.parametrize("spatial", [False, True])
def test_read_back_is_in_the_callers_order(ns_min, spatial):
    rng = np.random.default_rng(ns_min)
    lengths = [3, 256, 17, 16, 15, 129, 128]
    while sum(lengths) < ns_min:
        lengths.append(int(rng.integers(3, 60)))
    rng.shuffle(lengths)
    box = 400.0
    p = sc.params_init(box / 2, delta=1e-5, min_cell_length=4.0, seed=5)
    fil = make_filaments(_straight(lengths, ns_min, box))
    s = sc.FilamentSystem(p, fil, precision="mixed", spatial_order=spatial)
    r, rp, fr = s.sites()
    np.testing.assert_array_equal(r, fil.r)
    np.testing.assert_array_equal(rp, fil.r)
    assert not fr.any()
    # the end-to-end vectors are differences of positions, the centres sums
    # of at most 256 of them: 256 roundings of the largest
    e2e, com = s.filament_stats()
    x = fil.r.reshape(3, -1)
    off = fil.site_off
    np.testing.assert_array_equal(e2e, x[:, off[1:] - 1] - x[:, off[:-1]])
    want = np.add.reduceat(x, off[:-1], axis=1) / np.diff(off)
    np.testing.assert_allclose(com, want, rtol=0, atol=256 * 2.0 ** -52 * np.abs(x).max())
    # moved positions, per-bond values and random forces against the same
    # system in the caller's storage order
    ref = sc.FilamentSystem(p, fil, precision="mixed", spatial_order=False)
    for q in (s, ref):
        q.step(1)
    for a, b in zip(s.sites(), ref.sites()):
        # the packed lanes round alike in either order: no pair interacts
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(s.tensions(), ref.tensions())
    np.testing.assert_array_equal(s.dr_state(), ref.dr_state())
    for a, b in zip(s.bond_forces(), ref.bond_forces()):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-5 * max(1.0, np.abs(b).max()))
    s.close()
    ref.close()


# 8192 counters fit a block's local memory
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_theta_histogram_paths_agree(precision):
    lengths = [3, 4, 20, 66, 67, 256] * 30
    box = 500.0
    p = sc.params_init(box / 2, delta=1e-4, min_cell_length=4.0, seed=9)
    s = sc.FilamentSystem(p, make_filaments(_straight(lengths, 3, box)), precision=precision)
    s.step(6)
    local = s.theta_histogram(128, 64)
    wide = s.theta_histogram(128, 65)
    np.testing.assert_array_equal(local, wide[:64])
    want = np.array([sum(n - 2 > row for n in lengths) for row in range(65)])
    np.testing.assert_array_equal(wide.sum(axis=1), want)
    # a shape beyond the kept scratch: 64 bytes per bond
    nb = sum(lengths) - len(lengths)
    big = s.theta_histogram(128, nb // 16 + 1)
    np.testing.assert_array_equal(big[:65], wide)
    s.close()
