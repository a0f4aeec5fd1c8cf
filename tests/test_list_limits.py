"""Candidate lists that no capacity holds are refused: the sums of list
lengths, kept in 32 bits per block of bonds, never come out as a total that
fits, and the capacity asked for is then past the limit.  And the length from which a handle without a caller's launch
shape leaves the balanced pair kernel, and comes back to it."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("limits") / "limits.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"),
                    "-I" + os.path.join(HERE, "..", "simcore_amd", "csrc"),
                    os.path.join(HERE, "limits_host.cpp"), "-o", so], check=True)
    out = ctypes.CDLL(so)
    for name in ("max_candidates", "candidates_of", "grown_capacity"):
        getattr(out, name).restype = ctypes.c_int64
    out.kept_length.restype = ctypes.c_int32
    i64 = ctypes.c_int64
    out.kept_length.argtypes = out.candidates_of.argtypes = [i64]
    out.grown_capacity.argtypes = [i64, i64]
    return out


# bonds, all of them in each other's lists
@pytest.mark.parametrize("nb", [1000, 46000, 46341, 65536, 262145, 2097151, 2097152, 2097153,
                                2200000, 3145728, 4194304, 4194305, 6291456, 16777216, 2**31 - 1])
def test_crowded_lists_are_refused(lib, nb):
    limit = lib.max_candidates()
    deg, exact = nb - 1, nb * (nb - 1)
    full, rest = divmod(nb, 1024)  # blocks of four groups of 256 bonds
    total = full * lib.kept_length(1024 * deg) + lib.kept_length(rest * deg)
    need = lib.candidates_of(total)
    if exact <= 2 * limit:
        assert need == exact // 2 and lib.grown_capacity(10, need) >= need
    else:
        assert total > 2 * limit and need > limit
        assert lib.grown_capacity(10, need) > limit  # which the allocation refuses


def test_limit_itself(lib):
    limit = lib.max_candidates()
    assert lib.candidates_of(2 * limit) == limit
    assert lib.grown_capacity(limit // 2, limit) == limit
    assert lib.candidates_of(lib.kept_length(2**40)) == limit + 1
    assert lib.grown_capacity(limit, limit + 1) == limit + 1


@pytest.mark.parametrize("nb, line", [(2, 160), (32768, 160), (32769, 80), (65536, 80), (65537, 32),
                                      (131072, 32), (131073, 16), (199999, 16), (200000, 40),
                                      (2000000, 40)])
def test_pair_kernel_by_length(lib, nb, line):
    asked = lambda mean, now: lib.pair_balanced(ctypes.c_int64(nb), ctypes.c_double(mean), now)
    assert asked(0.0, 0) and asked(0.0, 1)
    assert asked(line, 1) and not asked(line * 1.001, 1)
    assert asked(0.75 * line, 0) and not asked(0.75 * line * 1.001, 0)
