"""Graphs of a batch replayed for other members: systems that agree in bonds,
sites, cells and packed waves but not in the number of filaments above 128
sites, which the integrator's grid depends on too."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.helpers import uneven_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first, second", [([200, 80, 20], [140, 140, 20]),
                                           ([140, 140, 20], [200, 80, 20])])
def test_members_with_other_long_filaments(first, second):
    cases = [uneven_system(sites=s, copies=1, radius=140.0, seed=5) for s in (first, second)]
    ens = sc.Ensemble(hbm_budget=2 << 30, max_active=1, steps_per_launch=16, batch_size=4)
    for p, f in cases:  # one after the other, in the same batch
        rid = ens.submit(p, f, 40, precision="mixed")
        ens.drain(60)
        with sc.FilamentSystem(p, f, precision="mixed", use_graph=True) as s:
            s.step(40)
            np.testing.assert_array_equal(ens.result(rid), s.sites()[0])
    assert ens.stats()["batched_steps"] == 80
    ens.close()
