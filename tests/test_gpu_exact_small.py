"""Random forces next to the least double: a caller's noise so small that the
right-hand sides of the random-force solve are below what a shared reciprocal
serves, or subnormal.  Value for value against the CPU path."""
import numpy as np
import pytest

import simcore_amd as sc
from oracle.oracle_py import OracleSystem
from tests.scenarios import make_filaments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponent", [-880, -905, -920, -1000, -1030, -1044, -1048, -1052, -1056,
                                      -1060, -1066])
def test_random_forces_of_any_size(exponent):
    rng = np.random.default_rng(7)
    sites = []
    for j, n in enumerate([3, 8, 20, 20, 33, 64, 130, 256]):
        u = np.cumsum(0.1 * rng.normal(size=(n - 1, 3)), axis=0) + [0, 0, 4.0]
        u /= np.linalg.norm(u, axis=1)[:, None]
        x = np.concatenate([np.zeros((1, 3)), np.cumsum(u, axis=0)])
        sites.append(x + [0, 40.0 * j - 140.0, -0.5 * n])
    p = sc.params_init(300.0, delta=1e-4, min_cell_length=4.0, seed=17)
    fil = make_filaments(sites)
    xi = np.ldexp(rng.uniform(-0.5, 0.5, 2 * 3 * fil.ns), exponent)
    dev = sc.FilamentSystem(p, fil, precision="fp64")
    ora = OracleSystem(p, fil)
    dev.set_noise(xi)
    ora.set_noise_buffer(xi, 2)
    for _ in range(3):
        dev.step(1)
        assert ora.step(1) == 0
        force = ora.sites()[2]
        assert force.any() and np.abs(force).max() < np.ldexp(1.0, exponent + 30)
        for a, b in zip(dev.sites(), ora.sites()):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(dev.tensions(), ora.tensions())
    dev.close()
    ora.close()
