"""The balanced pair kernel's bonds per wavefront (16, 32 or 64, by the number
of bonds) against the per-bond kernel, which adds the same shares in the same
order: bit for bit, at the edges of a wavefront and of the rule."""
import numpy as np
import pytest

import simcore_amd as sc
from tests.scenarios import make_filaments

pytestmark = pytest.mark.gpu


def _system(nb, precision, thermo):
    rng = np.random.default_rng(nb)
    half = max(6.0, 0.5 * (2.0 * nb) ** (1.0 / 3.0))
    p = sc.params_init(half, delta=1e-4, min_cell_length=2.0, seed=5)
    lengths, left = [], nb
    while left > 0:
        k = min(left, int(rng.integers(2, 40)))
        if left - k == 1:
            k += 1
        lengths.append(k + 1)
        left -= k
    u = rng.normal(size=(len(lengths), 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    start = rng.uniform(-half, half, (len(lengths), 3))
    fil = make_filaments([start[f] + np.arange(n)[:, None] * u[f]
                          for f, n in enumerate(lengths)])
    assert fil.nb == nb
    s = sc.FilamentSystem(p, fil, precision=precision, use_graph=True, spatial_order=True)
    if thermo:
        s.thermo_enable()
    return s


@pytest.mark.parametrize("thermo", [False, True])
@pytest.mark.parametrize("nb, precision", [
    (2, "fp64"), (15, "fp64"), (16, "fp64"), (17, "mixed"), (33, "mixed"), (65, "fp64"),
    (1000, "mixed"), (65536, "mixed"), (65537, "fp64"), (131072, "mixed"), (131073, "mixed")])
def test_split_matches_per_bond_kernel(nb, precision, thermo):
    a, b = _system(nb, precision, thermo), _system(nb, precision, thermo)
    layout = a.launch_shape()["integrate_layout"]
    assert a.launch_shape()["pair_block"] == 0
    b.set_launch_shape(pair_block=128, integrate_layout=layout)
    a.step(6)
    b.step(6)
    for x, y in zip(a.sites() + a.bond_forces(), b.sites() + b.bond_forces()):
        np.testing.assert_array_equal(x, y)
    if thermo:
        np.testing.assert_array_equal(a.bond_energies(), b.bond_energies())
        # sums of up to 3 nb terms of both signs: 3 nb roundings of the largest
        # partial sum, which the diagonal's magnitude stands for
        pa, pb = a.calculate_pressure(6), b.calculate_pressure(6)
        tol = 3 * nb * 2.0 ** -53 * max(1.0, np.abs(pb["pressure_tensor"]).max())
        np.testing.assert_allclose(pa["pressure_tensor"], pb["pressure_tensor"], rtol=0, atol=tol)
    a.close()
    b.close()
