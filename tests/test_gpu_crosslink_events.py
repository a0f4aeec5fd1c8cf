"""Rebinding at the edges of its lane split: one, two and many crosslinks of a
wavefront coming off in a step, last wavefronts with one lane, and per-bond
lists rebuilt by one and by several blocks (4096 bonds each), against the CPU
path value for value."""
import numpy as np
import pytest

import simcore_amd as sc
from oracle.oracle_py import OracleSystem
from tests.helpers import box_for_fraction

pytestmark = pytest.mark.gpu


# filaments, crosslinks, rate (a crosslink comes off with 1 - exp(-rate * dt))
@pytest.mark.parametrize("nf, nx, k_off", [
    (20, 1, 20000.0), (150, 63, 300.0), (150, 64, 600.0), (150, 65, 30000.0),
    (273, 700, 100.0), (274, 2000, 5000.0), (600, 1500, 200.0), (600, 3001, 30000.0)])
def test_rebinding_bit_exact(nf, nx, k_off):
    n = np.full(nf, 16, dtype=np.int32)
    p = sc.params_init(box_for_fraction(n, 1.0, 1.0, 0.08), delta=1e-4, min_cell_length=1.0,
                       seed=17)
    fil = sc.generate_filaments(p, n, 15.0, 50.0, 1.0, 2.0, seed=nf)
    b, lam = sc.generate_crosslinks(p, fil, nx, r_bind=2.0, seed=nx)
    xl = dict(k_spring=10.0, rest_length=1.0, k_compress=-1.0, k_off=k_off, r_bind=2.0, seed=99)
    dev = sc.FilamentSystem(p, fil, precision="fp64", use_graph=True)
    dev.load_crosslinks(b, lam, **xl)
    ora = OracleSystem(p, fil)
    ora.load_crosslinks(b, lam, **xl)
    for steps in (3, 9, 30):
        dev.step(steps)
        assert ora.step(steps) == 0
        db, dl, df, events = dev.crosslinks()
        ob, ol, of = ora.crosslinks()
        assert events == ora.xlink_events()
        np.testing.assert_array_equal(db, ob)
        np.testing.assert_array_equal(dl, ol)
        np.testing.assert_array_equal(df, of)
        for x, y in zip(dev.sites(), ora.sites()):
            np.testing.assert_array_equal(x, y)
    assert events > 0
