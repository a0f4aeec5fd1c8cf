"""The pair kernel that bench.py names, by precision, launch shape and size, and
its committed traffic, which is the entry of that kernel and no other's."""
import json
import os

import pytest

from tests.test_bench_cli import ROOT, _bench


@pytest.mark.parametrize("nb, bonds", [(992, 16), (65536, 16), (65537, 32), (131072, 32),
                                       (131073, 64), (1611162, 64)])
def test_pair_kernel_by_size(nb, bonds):
    B = _bench()
    assert B.pair_kernel(True, "mixed", nb) == f"k_pair_bal<true, false, {bonds}>"
    assert B.pair_kernel(True, "fp64", nb) == f"k_pair_bal<false, false, {bonds}>"
    assert B.pair_kernel(False, "mixed", nb) == "k_pair_fused<true, false>"


@pytest.mark.parametrize("tag, nb", [("uneven1600k_mixed", 1611162), ("dense620k_mixed", 620000)])
def test_traffic_is_of_the_kernel_named(tag, nb):
    B = _bench()
    with open(os.path.join(ROOT, "profiles", f"traffic_{tag}.json")) as fh:
        kernels = json.load(fh)["kernels"]
    name = B.pair_kernel(True, "mixed", nb)
    assert B.measured_traffic(tag, name) == kernels["sc::" + name]["traffic_bytes"]
    assert B.measured_traffic(tag, "k_pair_bal<true, false, 1>") is None
