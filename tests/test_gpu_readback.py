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
