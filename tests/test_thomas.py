"""The FP64 integrator's Thomas solve with shared reciprocals, compiled for the
host: where it says that it served, every value is the plain divisions' bit for
bit; right-hand sides of any size, down to the least double and up to where the
quotients overflow, either are served so or are left to the plain divisions."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
DP = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("thomas") / "thomas.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                    "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    "-I" + os.path.join(HERE, "..", "simcore_amd", "csrc"),
                    os.path.join(HERE, "thomas_host.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def _solve(lib, fast, diag, rhs, off):
    rows = np.ascontiguousarray(np.stack([diag, rhs], axis=1))
    off = np.ascontiguousarray(off)
    ok = lib.thomas(fast, len(rows), rows.ctypes.data_as(DP), off.ctypes.data_as(DP))
    return ok, rows


def _chain(rng, n, igpar=1.0, igperp=0.5):
    """Tension rows of a bent chain of n bonds."""
    u = np.cumsum(0.3 * rng.normal(size=(n, 3)), axis=0) + [0, 0, 3.0]
    u /= np.linalg.norm(u, axis=1)[:, None]
    t = np.vstack([u[:1], u[1:] + u[:-1], u[-1:]])
    t /= np.linalg.norm(t, axis=1)[:, None]
    a1, a2 = (t[:-1] * u).sum(1), (t[1:] * u).sum(1)
    diag = 2 * igperp + (igpar - igperp) * (a1 * a1 + a2 * a2)
    off = np.zeros(n)
    off[:-1] = -igperp * (u[1:] * u[:-1]).sum(1) - (igpar - igperp) * (a2[:-1] * a1[1:])
    return diag, off


# powers of two of the right-hand side; both ends of the doubles and the edges
# of the shared quotients' range
EXPONENTS = [-1074, -1073, -1060, -1050, -1044, -1043, -1042, -1041, -1040, -1030, -1023, -1022,
             -1021, -1000, -960, -901, -900, -899, -890, -500, -100, 0, 100, 500, 900, 1000, 1015,
             1020, 1021, 1022, 1023]


@pytest.mark.parametrize("exponent", EXPONENTS)
@pytest.mark.parametrize("frictions", [(1.0, 0.5), (2.0**15, 2.0**-4), (2.0**-48, 2.0**-30)])
def test_served_solves_equal_plain_divisions(lib, exponent, frictions):
    rng = np.random.default_rng(exponent + 2000)
    served = 0
    for n in (2, 3, 7, 31, 255):
        for one in (False, True):  # right-hand sides everywhere, or in one row
            diag, off = _chain(rng, n, *frictions)
            with np.errstate(over="ignore", under="ignore"):
                rhs = np.ldexp(rng.choice([-1, 1], n) * rng.uniform(1, 2, n), exponent)
            if one:
                rhs[np.arange(n) != rng.integers(n)] = 0.0
            ok, got = _solve(lib, 1, diag, rhs, off)
            _, want = _solve(lib, 0, diag, rhs, off)
            if ok:
                np.testing.assert_array_equal(got.view(np.uint64), want.view(np.uint64))
                served += 1
            else:  # only where the range ends
                assert exponent < -800 or not np.isfinite(want[:, 1]).all() or exponent > 950
    if -500 <= exponent <= 500:
        assert served == 10  # the plain divisions are not the usual path


def test_zero_right_hand_sides_are_served(lib):
    diag, off = _chain(np.random.default_rng(1), 40)
    for zero in (0.0, -0.0):
        ok, got = _solve(lib, 1, diag, np.full(40, zero), off)
        _, want = _solve(lib, 0, diag, np.full(40, zero), off)
        assert ok
        np.testing.assert_array_equal(got.view(np.uint64), want.view(np.uint64))


def test_overflowing_quotients_are_left_to_the_plain_divisions(lib):
    """A pivot below one turns a large right-hand side into an infinity in the
    first, a middle and the last row."""
    for at in (0, 20, 39):
        diag, off = np.full(40, 2.0**-8), np.full(40, -2.0**-10)
        off[-1] = 0.0
        rhs = np.zeros(40)
        rhs[at] = 2.0**1020
        assert not np.isfinite(_solve(lib, 0, diag, rhs, off)[1]).all()
        assert not _solve(lib, 1, diag, rhs, off)[0]


def test_frictions_served(lib):
    f = lambda a, b: lib.frictions(ctypes.c_double(a), ctypes.c_double(b))
    assert f(1.0, 0.5) and f(2.0**40, 2.0**25) and f(2.0**-49, 2.0**-35)
    for a, b in ((2.0**51, 2.0**51), (2.0**-51, 2.0**-51), (1.0, 2.0**21), (2.0**21, 1.0),
                 (0.0, 1.0), (1.0, float("nan")), (float("inf"), float("inf")), (-1.0, 1.0)):
        assert not f(a, b)
