"""A batch whose one-launch rebuild would take more blocks than pay (768): every
member is as when stepped alone on both sides of that line, in blocks of 512
(400 bonds each) and of 1024 threads (800 bonds each), members of equal and of
mixed sizes, and when a replayed batch changes sides."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.test_gpu_rebuild_launches import _fill

pytestmark = pytest.mark.gpu


def _alone(p, fil, steps):
    with sc.FilamentSystem(p, fil, precision="mixed", use_graph=True) as s:
        s.step(steps)
        assert s.counters()["n_rebuilds"] > 1
        return s.sites()[0]


def _sparse(nb):
    """Lists short enough for the one launch (16 entries a bond)."""
    return _fill(max(12, int(round((nb / 0.35) ** (1.0 / 3.0)))), nb, delta=1e-3)


# 768 and 769 blocks of either kind, some more of the smaller, and one large
# member among small ones
@pytest.mark.parametrize("bonds", [[38400] * 8, [38400] * 7 + [38402], [76800] * 8,
                                   [76800] * 7 + [76802], [33000] * 16, [90000] + [600] * 15])
def test_members_on_both_sides(bonds):
    made = {nb: _sparse(nb) for nb in set(bonds)}
    with sc.Ensemble(hbm_budget=16 << 30, max_active=16, steps_per_launch=16,
                     batch_size=16) as ens:
        for n in (len(bonds), len(bonds) // 2):  # the same batch, then half of it
            ids = []
            for k in range(n):
                p, fil = made[bonds[-1 - k]]
                assert fil.nb == bonds[-1 - k]
                p.seed = k + 1
                ids.append(ens.submit(p, fil, 41, precision="mixed"))
            ens.drain(60)
            for k in (0, n // 2, n - 1):
                p, fil = made[bonds[-1 - k]]
                p.seed = k + 1
                np.testing.assert_array_equal(ens.result(ids[k]), _alone(p, fil, 41))
        assert ens.stats()["batched_steps"] > 0
