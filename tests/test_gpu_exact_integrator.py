"""The FP64 integrator against the CPU path, value for value: filament sizes
at the edges of its slices and blocks, several bins in one launch, and
frictions outside the range its shared reciprocals serve."""
import numpy as np
import pytest

import simcore_amd as sc
from oracle.oracle_py import OracleSystem
from tests.scenarios import make_filaments

pytestmark = pytest.mark.gpu


def _bent(lengths, seed, box=600.0):
    """Gently bent filaments, too far apart to interact."""
    rng = np.random.default_rng(seed)
    out = []
    for j, n in enumerate(lengths):
        u = rng.normal(size=3)
        x = np.empty((n, 3))
        x[0] = rng.uniform(-0.5, 0.5, 3) * box
        for i in range(1, n):
            u = u / np.linalg.norm(u) + 0.2 * rng.normal(size=3)
            u /= np.linalg.norm(u)
            x[i] = x[i - 1] + u
        out.append(x)
    return out


def _compare(lengths, steps=6, gamma=None, delta=1e-5, lp=50.0):
    p = sc.params_init(300.0, delta=delta, min_cell_length=4.0, seed=17)
    fil = make_filaments(_bent(lengths, len(lengths)), lp=lp)
    if gamma is not None:
        for f in fil.fil:
            f.gamma_perp, f.gamma_par = gamma, 0.5 * gamma
    dev = sc.FilamentSystem(p, fil, precision="fp64")
    ora = OracleSystem(p, fil)
    dev.step(steps)
    assert ora.step(steps) == 0
    for a, b in zip(dev.sites(), ora.sites()):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(dev.tensions(), ora.tensions())
    assert np.isfinite(dev.tensions()).all() and dev.tensions().any()
    dev.close()
    ora.close()


# sites per filament and filaments: fewer, exactly and more than a block's
@pytest.mark.parametrize("n", [3, 4, 5, 6, 8, 9, 16, 17, 33, 64, 65, 85, 86, 127, 128, 129, 255,
                               256])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_equal_lengths(n, extra):
    per = min(64, 256 // n, 288 // (n | 1))
    _compare([n] * max(1, per + extra))


def test_every_bin_in_one_launch():
    rng = np.random.default_rng(4)
    lengths = [3, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 256] + rng.integers(3, 257, 60).tolist()
    _compare(lengths, steps=9)


# outside [2^-50, 2^50]; the time step keeps the displacements ordinary
@pytest.mark.parametrize("gamma, delta", [(2e15, 1e9), (1e-17, 1e-22)])
def test_frictions_outside_the_shared_reciprocal(gamma, delta):
    _compare([3, 20, 40, 256], gamma=gamma, delta=delta)
