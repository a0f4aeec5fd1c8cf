"""Candidate lists where the rebuild's launches change shape: numbers of cell
columns at the edges of a scan tile (4096) and of the one-launch scan (2^17),
numbers of bonds at the edges of the list pass's groups (256) and blocks of
groups (1024).  Checked against a brute-force walk over all pairs."""
import numpy as np
import pytest

import simcore_amd as sc
from oracle.oracle_py import OracleSystem
from tests.scenarios import make_filaments

pytestmark = pytest.mark.gpu


def _system(n1d, nb, seed):
    """Straight filaments with nb bonds in all in a box of n1d cells of side 2,
    in a few clumps so that lists are not empty."""
    rng = np.random.default_rng(seed)
    box = 2.0 * n1d
    lengths = []
    left = nb
    while left > 0:
        k = min(left, int(rng.integers(2, 40)))
        if left - k == 1:
            k += 1
        lengths.append(k + 1)
        left -= k
    sites = []
    for n in lengths:
        u = rng.normal(size=3)
        u /= np.linalg.norm(u)
        start = (rng.integers(0, 3, 3) / 3.0 - 0.5) * box + rng.normal(size=3) * 6.0
        sites.append(start + np.arange(n)[:, None] * u)
    p = sc.params_init(box / 2, delta=1e-6, min_cell_length=2.0, seed=3)
    return p, make_filaments(sites)


def _brute(keys, n, site_off):
    c = np.stack([keys // (n * n), keys // n % n, keys % n])
    near = np.ones((len(keys), len(keys)), bool)
    for x in c:
        d = (x[:, None] - x[None, :]) % n
        near &= (d <= 1) | (d == n - 1)
    i, j = np.nonzero(np.triu(near, 1))
    fil = np.repeat(np.arange(len(site_off) - 1), np.diff(site_off) - 1)
    keep = ~((j - i == 1) & (fil[i] == fil[j]))
    return set(zip(i[keep].tolist(), j[keep].tolist()))


@pytest.mark.parametrize("n1d, nb", [(63, 255), (64, 256), (65, 257), (90, 511), (91, 513),
                                     (362, 300), (363, 300), (40, 8191), (40, 8192), (40, 8193),
                                     (363, 1023), (363, 1024), (363, 1025)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lists_at_launch_edges(n1d, nb, precision):
    p, fil = _system(n1d, nb, n1d + nb)
    assert fil.nb == nb
    s = sc.FilamentSystem(p, fil, precision=precision, use_graph=True)
    assert s.counters()["n_cells_1d"] == n1d
    a, b = s.candidates()
    got = set(zip(np.minimum(a, b).tolist(), np.maximum(a, b).tolist()))
    assert len(got) == len(a)
    assert got == _brute(s.cell_keys().astype(np.int64), n1d, np.asarray(fil.site_off))
    s.step(4)
    s.close()


def _cell_pairs(keys, n, site_off):
    """Sorted pair codes (a * nb + b, a < b) of the bonds in adjacent cells,
    neighbours along a filament left out, cell by cell."""
    nb = len(keys)
    order = np.argsort(keys, kind="stable")
    ks = keys[order]
    c = np.stack([ks // (n * n), ks // n % n, ks % n])
    fil = np.repeat(np.arange(len(site_off) - 1), np.diff(site_off) - 1)
    out = []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dz in (-1, 0, 1):
                m = [(c[0] + dx) % n, (c[1] + dy) % n, (c[2] + dz) % n]
                kk = (m[0] * n + m[1]) * n + m[2]
                lo, hi = np.searchsorted(ks, kk), np.searchsorted(ks, kk, side="right")
                cnt = hi - lo
                i = np.repeat(np.arange(nb), cnt)
                j = np.arange(len(i)) - np.repeat(np.cumsum(cnt) - cnt, cnt) + np.repeat(lo, cnt)
                a, b = order[i], order[j]
                keep = (a < b) & ~((b - a == 1) & (fil[a] == fil[b]))
                out.append(a[keep].astype(np.int64) * nb + b[keep])
    return np.sort(np.concatenate(out))


def _spread(nb):
    """(params, filaments, cells a side): straight filaments with nb bonds in
    all, anywhere in the box."""
    rng = np.random.default_rng(nb)
    n1d = max(12, int(round((nb / 1.5) ** (1.0 / 3.0))))
    p = sc.params_init(float(n1d), delta=1e-4, min_cell_length=2.0, seed=11)
    lengths, left = [], nb
    while left > 0:
        k = min(left, int(rng.integers(2, 60)))
        if left - k == 1:
            k += 1
        lengths.append(k + 1)
        left -= k
    u = rng.normal(size=(len(lengths), 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    start = rng.uniform(-n1d, n1d, (len(lengths), 3))
    fil = make_filaments([start[f] + np.arange(n)[:, None] * u[f]
                          for f, n in enumerate(lengths)])
    return p, fil, n1d


# 400 and 800 bonds a block of the one-launch rebuild, which has blocks of 512
# threads up to 40960 bonds and serves 262144
@pytest.mark.parametrize("nb", [799, 800, 801, 25599, 40960, 40961, 102401, 131073, 262143, 262144, 262145])
def test_lists_of_one_and_several_launches(nb):
    p, fil, n1d = _spread(nb)
    assert fil.nb == nb
    s = sc.FilamentSystem(p, fil, precision="mixed", use_graph=True, spatial_order=True)
    assert s.counters()["n_cells_1d"] == n1d
    for steps in (0, 41):  # the list of the load, then of rebuilds inside a run
        s.step(steps)
        a, b = s.candidates()
        code = np.sort(np.minimum(a, b).astype(np.int64) * nb + np.maximum(a, b))
        want = _cell_pairs(s.cell_keys().astype(np.int64), n1d, np.asarray(fil.site_off))
        np.testing.assert_array_equal(code, want)
    assert s.counters()["n_rebuilds"] > 1
    s.close()


# cells around a bond: few, about the 12 that a bond's slab of runs holds, all
# 27; `clump` bonds more in one cell, about the 255 that a slab's length holds
@pytest.mark.parametrize("n1d, nb, clump", [(12, 300, 0), (12, 700, 0), (12, 1100, 0), (3, 600, 0),
                                            (12, 400, 252), (12, 400, 254), (12, 400, 256),
                                            (5, 800, 400)])
def test_lists_at_the_edges_of_a_slab(n1d, nb, clump):
    rng = np.random.default_rng(100 * n1d + nb + clump)
    p = sc.params_init(float(n1d), delta=1e-4, min_cell_length=2.0, seed=11)
    bonds = [rng.uniform(-n1d, n1d, 3) for _ in range(nb // 2)]  # two bonds each, straight
    bonds += [1.0 + rng.uniform(-0.3, 0.3, 3) - n1d % 2 for _ in range(clump // 2)]
    u = rng.normal(size=(len(bonds), 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    step = np.where(np.arange(len(bonds)) < nb // 2, 1.0, 0.1)
    sites = [c + np.arange(-1, 2)[:, None] * w * s for c, w, s in zip(bonds, u, step)]
    fil = make_filaments(sites)
    s = sc.FilamentSystem(p, fil, precision="fp64")
    a, b = s.candidates()
    code = np.sort(np.minimum(a, b).astype(np.int64) * fil.nb + np.maximum(a, b))
    keys = s.cell_keys().astype(np.int64)
    if clump:
        assert np.bincount(keys).max() >= clump - 2
    np.testing.assert_array_equal(code, _cell_pairs(keys, n1d, np.asarray(fil.site_off)))
    # the order of each list, by the sums it gives
    ora = OracleSystem(p, fil)
    s.step(2)
    assert ora.step(2) == 0
    for x, y in zip(s.bond_forces(), ora.bond_forces()):
        np.testing.assert_array_equal(x, y)
    s.close()


def test_batch_of_more_blocks_than_fit():
    """The one-launch rebuild of 24 members asks for more blocks than the chip
    holds, so members start their passes with some of theirs."""
    p, fil, _ = _spread(40000)
    seeds = list(range(1, 25))
    ens = sc.Ensemble(hbm_budget=16 << 30, max_active=24, steps_per_launch=16, batch_size=24)
    ids = []
    for k in seeds:
        p.seed = k
        ids.append(ens.submit(p, fil, 41, precision="mixed"))
    ens.drain(60)
    for k in (1, 9, 17, 24):
        p.seed = k
        s = sc.FilamentSystem(p, fil, precision="mixed", use_graph=True)
        s.step(41)
        assert s.counters()["n_rebuilds"] > 1
        np.testing.assert_array_equal(ens.result(ids[k - 1]), s.sites()[0])
        s.close()
    ens.close()


def test_batch_with_a_wide_member():
    """A batch member with more columns than the one-launch scan takes, beside
    a small one: each as when stepped alone."""
    cases = [_system(363, 300, 5), _system(40, 600, 6)]
    for p, _ in cases:
        p.delta = 1e-4
    ens = sc.Ensemble(hbm_budget=4 << 30, max_active=4, steps_per_launch=16, batch_size=4)
    ids = [ens.submit(p, f, 40, precision="mixed") for p, f in cases]
    ens.drain(60)
    for i, (p, f) in zip(ids, cases):
        s = sc.FilamentSystem(p, f, precision="mixed", use_graph=True)
        s.step(40)
        np.testing.assert_array_equal(ens.result(i), s.sites()[0])
        s.close()
    ens.close()
