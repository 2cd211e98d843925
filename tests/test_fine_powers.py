"""The land-surface step's power and logarithm (pow_fine and ln_fine, built into the library
for host and device from one source) against 80-bit arithmetic, over the step's ranges and
past them.

They stand where the reference calls libm's pow and log (src/noah/noah.c), so they have to
be as accurate as a C library's.  The bound is derived: ln x is carried to 3e-18 of its
size, so y ln x brings |y ln x| 3e-18 to the result; in e^r the quadratic and higher terms,
at most 0.061, round at 1.5 ulp of their own and once more in the last sum (0.2 ulp of the
result together) and the result itself rounds by half an ulp."""
import numpy as np
import pytest

from pihm_amd import _lib

LD = np.longdouble


def _fine(x, y=None, device=False):
    x = np.ascontiguousarray(x, dtype=np.float64)
    y = None if y is None else np.ascontiguousarray(np.broadcast_to(y, x.shape), dtype=np.float64)
    out = np.empty_like(x)
    dp = lambda a: None if a is None else a.ctypes.data_as(_lib.c_double_p)
    assert _lib.lib().pihm_math_fine(len(x), dp(x), dp(y), dp(out), 1 if device else 0) == 0
    return out


def _cases(n=40000):
    rng = np.random.default_rng(7)
    u = rng.uniform
    return {
        "friction velocity": (10 ** u(-30, 4, n), np.full(n, 2.0 / 3.0)),
        "snow density": (u(1e-3, 60.0, n), np.full(n, 1.5)),
        "snow conductivity": (np.full(n, 10.0), u(0.0, 3.0, n)),
        "snow age": (np.full(n, 0.94), u(0.0, 60.0, n)),
        "age": (10 ** u(-3, 3, n), np.full(n, 0.58)),
        "evaporation": (10 ** u(-12, 0, n), u(0.5, 3.0, n)),
        "minerals": (np.full(n, 7.7), u(0.0, 1.0, n)),
        "frozen water": (u(0.01, 1.0, n), -u(1.1, 21.0, n)),
        "frozen water head": (10 ** u(-6, 6, n), u(1.05, 4.0, n)),
        "frozen water root": (10 ** u(-6, 6, n), -u(0.05, 0.95, n)),
        "near one": (1.0 - 10 ** u(-16, -1, n), u(-21.0, 21.0, n)),
        "whole range": (10 ** u(-300, 300, n), u(-1.0, 1.0, n)),
    }


def _ulps(got, ref):
    return np.abs((got.astype(LD) - ref) / np.spacing(np.abs(ref.astype(np.float64)))).astype(float)


@pytest.mark.parametrize("name", list(_cases(1)))
def test_power_within_its_bound(name):
    x, y = _cases()[name]
    t = np.abs(y.astype(LD) * np.log(x.astype(LD))).astype(float)
    ref = x.astype(LD) ** y.astype(LD)
    e = _ulps(_fine(x, y), ref)
    # relative errors of |t| 3e-18 and of the 80-bit power itself are up to 2^53 times that in ulps
    assert np.all(e <= 0.7 + t * 3.0e-18 * 2.0 ** 53)
    assert e.mean() <= 0.26        # rounding alone: 0.25


def test_logarithm_within_its_bound():
    rng = np.random.default_rng(8)
    n = 100000
    for x in (10 ** rng.uniform(-307, 307, n), 1.0 + rng.choice([-1, 1], n) * 10 ** rng.uniform(-15.5, -0.4, n),
              rng.uniform(0.3, 3.0, n), np.array([5e-324, 1e-310, 2.0 ** -1022, 1.7e308])):
        assert np.all(_ulps(_fine(x), np.log(x.astype(LD))) <= 0.53)


def test_special_arguments_follow_libm():
    v = np.array([0.0, -0.0, 1.0, -1.0, 2.0, -2.0, 0.5, -0.5, 3.0, -3.0, 1e300, -1e300, 1e-300, np.inf, -np.inf, np.nan])
    x, y = (a.ravel() for a in np.meshgrid(v, v))
    with np.errstate(all="ignore"):
        for got, ref in ((_fine(x, y), np.power(x, y)), (_fine(v), np.log(v))):
            plain = np.isfinite(ref) & (ref != 0.0)
            assert np.array_equal(got[~plain], ref[~plain], equal_nan=True)
            assert np.array_equal(np.signbit(got[~np.isnan(ref)]), np.signbit(ref[~np.isnan(ref)]))
            assert np.allclose(got[plain], ref[plain], rtol=2.0 ** -52, atol=0.0)


def test_powers_past_the_range():
    rng = np.random.default_rng(4)
    x = 10 ** rng.uniform(-300, 300, 20000)
    y = np.log(10.0) * rng.choice([-1, 1], 20000) * rng.uniform(306, 330, 20000) / np.log(x)
    got = _fine(x, y)
    with np.errstate(over="ignore", under="ignore"):
        ref = (x.astype(LD) ** y.astype(LD)).astype(np.float64)
    fin = np.isfinite(ref) & np.isfinite(got)
    # the rounding of y ln x (710 3e-18) is up to 19 ulp here; subnormal results add one step
    assert np.all(np.abs(got[fin] - ref[fin]) <= 20 * np.spacing(np.abs(ref[fin])) + 1e-323)
    assert np.array_equal(np.isfinite(ref), np.isfinite(got))


@pytest.mark.gpu
def test_device_returns_the_host_bits():
    for name, (x, y) in _cases(20000).items():
        print(f"[fine] {name}", flush=True)
        assert np.array_equal(_fine(x, y), _fine(x, y, device=True))
        assert np.array_equal(_fine(x), _fine(x, device=True))
